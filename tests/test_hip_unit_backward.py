"""The reverse pass of heads spread over compute units by unit (float32 beyond head dim 64, bf16 beyond 128) at the edges of
its members (16 or 32 units), row tiles (4, 8, 16 rows), bursts (8, 4, 2 steps) and launches, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import slstm_oracle as so
from tests._util import geometric_reset_mask, make_problem, r_ext_to_kernel

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _problem(bf16, B, T, NH, dh, masked):
    H = NH * dh
    wx, r, b, s0 = make_problem(700 + dh, B, T, NH, dh, rscale=2.0, bf16=bf16, with_state=masked)
    reset = geometric_reset_mask(dh, B, T, max(2, T // 3)) if masked else None
    rng = np.random.default_rng(dh)
    d_h = rng.standard_normal((T, B, H)).astype(np.float32)
    d_sf = rng.standard_normal((4, B, H)).astype(np.float32)
    d_sf[3] = 0.0
    dt = torch.bfloat16 if bf16 else torch.float32
    if bf16:
        d_h = torch.from_numpy(d_h).bfloat16().float().numpy()
        r = torch.from_numpy(r).bfloat16().float().numpy()
    t = lambda x: None if x is None else torch.from_numpy(x).to(DEV)
    dev = (t(wx).to(dt), r_ext_to_kernel(torch.from_numpy(r)).to(DEV), t(b), t(s0) if masked else None, t(reset))
    # the gradient of h as a layer's norm hands it back: [B, S, H] in memory
    return (wx, r, b, s0, reset, d_h, d_sf), dev, t(d_h).to(dt).transpose(0, 1).contiguous().transpose(0, 1), t(d_sf)


@pytest.mark.parametrize("bf16,B,T,NH,dh,masked,opts", [
    (False, 1, 1, 1, 72, False, {}), (False, 5, 17, 2, 72, True, {}), (False, 4, 9, 3, 136, True, {}), (False, 9, 18, 4, 264, True, {}),
    (False, 40, 6, 4, 264, True, {}), (False, 3, 8, 9, 512, False, {}), (False, 6, 11, 2, 96, True, dict(recurrent_clipval=0.05)),
    (True, 1, 2, 1, 136, False, {}), (True, 4, 17, 3, 200, True, {}), (True, 21, 16, 4, 200, True, {}), (True, 5, 9, 2, 320, True, {}),
    (True, 3, 10, 1, 520, True, {}), (True, 20, 7, 2, 520, True, {}), (True, 20, 6, 8, 520, True, {}), (True, 2, 5, 9, 520, False, {}),
    (True, 7, 9, 1, 1000, True, {}), (True, 9, 7, 4, 1024, True, {}), (True, 5, 11, 2, 144, True, dict(recurrent_cut=True)),
])
def test_unit_backward_against_the_oracle(bf16, B, T, NH, dh, masked, opts):
    from xlstm_amd import functional as F

    print("case unit backward", bf16, B, T, NH, dh, masked, opts, flush=True)
    host, dev, d_h, d_sf = _problem(bf16, B, T, NH, dh, masked)
    coef = F.training_coefficients(dev[0], NH)
    h, s = F.slstm_forward(*dev, train_coef=coef)
    h_plain, s_plain = F.slstm_forward(*dev)
    assert torch.equal(h, h_plain) and torch.equal(s, s_plain)
    o = so.slstm_backward(*host, **opts)
    o = (o[0], r_ext_to_kernel(torch.from_numpy(o[1])).numpy(), o[2], o[3])
    for c in (coef, None):
        got = F.slstm_backward(*dev, h, d_h, d_sf, coef=c, **opts)
        errs = [float(np.abs(x.cpu().numpy() - y).max() / max(1.0, np.abs(y).max())) for x, y in zip(got, o)]
        print(errs, flush=True)
        assert all(np.isfinite(e) and e <= (2e-2 if bf16 else 1e-5) for e in errs), errs
    if bf16:
        short = F.slstm_backward(*dev, h, d_h, d_sf, coef=coef, d_wx_dtype=torch.bfloat16, **opts)
        assert torch.equal(short[0], got[0].bfloat16()) and torch.equal(short[3], got[3])


@pytest.mark.parametrize("bf16,B,NH,dh", [(False, 5, 2, 96), (True, 5, 1, 520)])
def test_a_wait_that_runs_out_is_reported(bf16, B, NH, dh):
    from xlstm_amd import functional as F

    _, dev, d_h, d_sf = _problem(bf16, B, 6, NH, dh, False)
    coef = F.training_coefficients(dev[0], NH)
    h, _ = F.slstm_forward(*dev, train_coef=coef)
    with pytest.raises(F.EngineError):
        F.slstm_backward(*dev, h, d_h, d_sf, coef=coef, spin_limit=-1)


@pytest.mark.parametrize("B,T,NH,dh", [(32, 256, 4, 1024), (12, 128, 8, 640)])
def test_no_wait_goes_on_until_the_abort_word_is_read(B, T, NH, dh):
    """Row tiles of 16 rows, head dims beyond 512: every wait ends with a look at the deltas, long before the 256th, behind which a
    wave reads the abort word (16 looks suffice; a line left in the vector cache had waves wait for that)."""
    from xlstm_amd import functional as F

    print("case looks", B, T, NH, dh, flush=True)
    H = NH * dh
    torch.manual_seed(dh)
    wx = torch.randn(B, T, 4 * H, device=DEV, dtype=torch.bfloat16)
    r = ((torch.rand(NH, 4 * dh, dh, device=DEV) * 2 - 1) / H ** 0.5).bfloat16()
    b = torch.zeros(NH, 4, dh, device=DEV)
    d_h = torch.randn(T, B, H, device=DEV).bfloat16()
    coef = F.training_coefficients(wx, NH)
    h, _ = F.slstm_forward(wx, r, b, train_coef=coef)
    want = F.slstm_backward(wx, r, b, None, None, h, d_h, coef=coef, d_wx_dtype=torch.bfloat16)
    for _ in range(5):
        got = F.slstm_backward(wx, r, b, None, None, h, d_h, coef=coef, d_wx_dtype=torch.bfloat16, spin_limit=200)
        assert torch.equal(got[0], want[0]) and torch.equal(got[3], want[3])
