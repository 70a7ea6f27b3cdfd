"""The tiled kernel of the gate projections at the edges of its tiles and of the rules that choose them: token counts
around 16-, 64- and 128-token tiles, one and several slabs of K, the placement of weights or tokens on one XCD."""
import pytest
import torch

from tests._util import max_err

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("NH,dh", [(1, 64), (3, 192), (4, 320), (2, 512), (4, 1024), (16, 64)])
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 577])
def test_gate_projections_at_tile_edges(NH, dh, M):
    from xlstm_amd import functional as hipF

    print("case gate tiles", NH, dh, M, flush=True)
    g = torch.Generator(device=DEV).manual_seed(M * 1000 + dh)
    H = NH * dh
    x, xc = (torch.randn(M, 1, H, device=DEV, generator=g).bfloat16() for _ in range(2))
    ws = [(torch.randn(NH, dh, dh, device=DEV, generator=g) * dh ** -0.5).bfloat16() for _ in range(4)]
    out = torch.full((M + 1, 1, 4 * H), 7.0, device=DEV, dtype=torch.bfloat16)  # (one row more: nothing may be written there)
    hipF.headwise_gates(x, xc, ws, NH, out=out[:M])
    torch.cuda.synchronize()
    assert bool((out[M] == 7.0).all())
    for s in range(4):
        a = (xc if s < 2 else x).float().view(M, NH, dh).transpose(0, 1).contiguous()
        want = torch.matmul(a, ws[s].float().transpose(1, 2).contiguous()).transpose(0, 1).reshape(M, H)
        assert max_err(out[:M].view(M, 4, H)[:, s].float().cpu().numpy(), want.cpu().numpy()) <= 2e-2
