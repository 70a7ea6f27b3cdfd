"""Training calls of a cell through the native host path against the Python one (which a replaced
``functional.slstm_backward`` takes): every layout of input and output, states, masks, options, gradients of any strides."""
import pytest
import torch

from tests._util import geometric_reset_mask

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype,in_shape,out_shape,B,T,NH,dh,extra", [
    (torch.float32, "BSGNH", "BNSH", 3, 7, 2, 64, {}), (torch.bfloat16, "BSGNH", "BSH", 5, 9, 2, 128, dict(state=True, mask=True)),
    (torch.float32, "SBGNH", "SBH", 2, 5, 3, 96, dict(state=True)), (torch.bfloat16, "SBGNH", "SBNH", 1, 2, 1, 200, dict(mask=True)),
    (torch.bfloat16, "BSGNH", "BNSH", 4, 6, 2, 136, dict(state=True, clip=1.0)), (torch.float32, "BSGNH", "BSH", 9, 4, 4, 256, dict(cut=True, mask=True)),
    (torch.bfloat16, "BSGNH", "BNSH", 2, 3, 2, 512, dict(bf16_params=True, state=True)),
])
def test_native_training_call_equals_the_python_path(monkeypatch, dtype, in_shape, out_shape, B, T, NH, dh, extra):
    from xlstm_amd import cell as cell_module
    from xlstm_amd.cell import sLSTMCell, sLSTMCellConfig

    print("case native training", dtype, in_shape, out_shape, B, T, NH, dh, extra, flush=True)
    torch.manual_seed(B * dh)
    H = NH * dh
    cell = sLSTMCell(sLSTMCellConfig(hidden_size=H, num_heads=NH, backend="hip", recurrent_weight_init="standard", input_shape=in_shape,
                                     output_shape=out_shape, gradient_recurrent_cut=bool(extra.get("cut")),
                                     gradient_recurrent_clipval=extra.get("clip"))).to(DEV)
    if extra.get("bf16_params"):
        cell = cell.bfloat16()
    x0 = torch.randn(B, T, 4 * H, device=DEV).to(dtype)
    x0 = x0 if in_shape == "BSGNH" else x0.transpose(0, 1).contiguous()
    s0 = torch.randn(4, B, H, device=DEV)
    s0[2] = s0[2].abs() + 1.0
    mask = torch.from_numpy(geometric_reset_mask(1, B, T, 3)).to(DEV).bool() if extra.get("mask") else None
    grads = None
    for wide in (False, True):  # gradients of the output as they come, and with strides that no kernel reads
        results = []
        for native in (True, False):
            if not native:
                plain = cell_module.F_hip.slstm_backward
                monkeypatch.setattr(cell_module.F_hip, "slstm_backward", lambda *a, **kw: plain(*a, **kw))
            x = x0.clone().requires_grad_(True)
            st = s0.to(dtype).requires_grad_(True) if extra.get("state") else None
            out, state = cell(x, st, reset_mask=mask)
            assert ("sLSTMCell" in out.grad_fn.name()) == native
            if grads is None:
                grads = torch.randn(*out.shape, 2, device=DEV).to(dtype), torch.randn_like(state)
            g = grads[0][..., 1] if wide else grads[0][..., 0].contiguous()
            leaves = [x, *cell.parameters()] + ([st] if st is not None else [])
            results.append([out, state, *torch.autograd.grad((out, state), leaves, (g, grads[1]), retain_graph=native)])
            if native:  # the graph once more, the gradient of the output alone
                results[0] += list(torch.autograd.grad(out, leaves, g))
            else:
                results[1] += list(torch.autograd.grad(cell(x, st, reset_mask=mask)[0], leaves, g))
            monkeypatch.undo()
        for i, (a, b) in enumerate(zip(*results)):
            assert a.shape == b.shape and a.dtype == b.dtype
            # (d R and d bias are summed with float atomics: not the same bits from run to run)
            torch.testing.assert_close(a, b, rtol=2e-2 if a.dtype == torch.bfloat16 else 1e-4, atol=2e-2 if a.dtype == torch.bfloat16 else 1e-4)
            if a.shape == x0.shape or i < 2:
                assert torch.equal(a, b), i
    with pytest.raises(RuntimeError, match="second time"):
        out, _ = cell(x, reset_mask=mask)
        torch.autograd.grad(out, x, torch.ones_like(out))
        torch.autograd.grad(out, x, torch.ones_like(out))
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out, _ = cell(x, reset_mask=mask)
        with torch.no_grad():
            cell._recurrent_kernel_.mul_(1.0)
        torch.autograd.grad(out, x, torch.ones_like(out))
