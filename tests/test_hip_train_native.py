"""Training calls of a cell through the native host path against the Python one (the tests replace the cell's choice
between them): every layout of input and output, states, masks, options, gradients of any strides."""
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
                monkeypatch.setattr(cell_module.sLSTMCell_hip, "_trains_natively", lambda self, input: False)
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


def _small_cell(NH=2, dh=64):
    from xlstm_amd.cell import sLSTMCell, sLSTMCellConfig

    torch.manual_seed(dh)
    cell = sLSTMCell(sLSTMCellConfig(hidden_size=NH * dh, num_heads=NH, backend="hip", recurrent_weight_init="standard")).to(DEV)
    return cell, torch.randn(3, 5, 4 * NH * dh, device=DEV, requires_grad=True)


def test_forward_mode_is_refused():
    print("case forward mode", flush=True)
    cell, x = _small_cell()
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        with pytest.raises((RuntimeError, NotImplementedError)):
            cell(dual)


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("dh", [64, 128])
def test_checkpointing_and_hooks_see_what_is_saved(monkeypatch, native, dh):
    """Checkpointing keeps nothing of the first forward; hooks pack the coefficients as well; gradients stay the same."""
    from torch.utils.checkpoint import checkpoint

    from xlstm_amd import cell as cell_module

    print("case saved tensors", native, dh, flush=True)
    if not native:
        monkeypatch.setattr(cell_module.sLSTMCell_hip, "_trains_natively", lambda self, input: False)
    cell, x = _small_cell(dh=dh)
    leaves = [x, *cell.parameters()]
    out, _ = cell(x)
    d = torch.randn_like(out)
    want = torch.autograd.grad(out, leaves, d)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.numel()), t.cpu())[1], lambda t: t.to(DEV)):
        hooked = torch.autograd.grad(cell(x)[0], leaves, d)
    coef = cell_module.F_hip.training_coefficients(x, 2).numel()
    assert coef in packed and x.numel() in packed and cell._bias_.numel() in packed
    again = torch.autograd.grad(checkpoint(lambda v: cell(v)[0], x, use_reentrant=False), leaves, d)
    for a, b, c in zip(want, hooked, again):
        # (sums over rows and steps by float atomics: 15 terms of order 1)
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(a, c, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("which", ["input", "_bias_", "_recurrent_kernel_"])
def test_changes_in_front_of_the_backward_are_refused(which):
    print("case in place", which, flush=True)
    cell, leaf = _small_cell()
    x = leaf * 1.0
    out, _ = cell(x)
    with torch.no_grad():
        (x if which == "input" else getattr(cell, which)).mul_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


@pytest.mark.parametrize("dtype,dh", [(torch.bfloat16, 64), (torch.float32, 96), (torch.bfloat16, 256), (torch.bfloat16, 512)])
def test_coefficients_beyond_what_is_kept(monkeypatch, dtype, dh):
    """Coefficients of a size that is not kept: the backward call makes them again, in slices of rows."""
    from xlstm_amd import cell as cell_module

    print("case coefficients not kept", dtype, dh, flush=True)
    cell, _ = _small_cell(dh=dh)
    B, T = 37, 4
    x = torch.randn(B, T, 8 * dh, device=DEV).to(dtype).requires_grad_(True)
    state = torch.randn(4, B, 2 * dh, device=DEV)
    state[2] = state[2].abs() + 1.0
    state = state.to(dtype).requires_grad_(True)
    mask = torch.from_numpy(geometric_reset_mask(1, B, T, 3)).to(DEV).bool()
    leaves = [x, state, *cell.parameters()]
    out, _ = cell(x, state, reset_mask=mask)
    d = torch.randn_like(out)
    want = torch.autograd.grad(out, leaves, d)
    for bound in ("KEPT_COEFFICIENT_BYTES", "RECOMPUTED_COEFFICIENT_BYTES"):
        monkeypatch.setattr(cell_module.F_hip, bound, 36 * T * 2 * dh * 16)
    out2, _ = cell(x, state, reset_mask=mask)
    assert torch.equal(out, out2) and "sLSTMCell" not in out2.grad_fn.name()
    for a, b in zip(want, torch.autograd.grad(out2, leaves, d)):
        # (row tiles of other heights sum in another order, and bfloat16 deltas round once: 2^-8)
        tol = 2e-2 if dtype == torch.bfloat16 else 1e-4
        torch.testing.assert_close(a, b, rtol=tol, atol=tol)


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("dtype,dh", [(torch.float32, 64), (torch.bfloat16, 128), (torch.bfloat16, 256)])
def test_a_stack_keeps_what_a_device_may_hold(monkeypatch, native, dtype, dh):
    """Four layers one behind the other and room for the coefficients of two: the others are made again by their backward
    calls, the gradients are the same, and everything is given back - behind the backward, and where none is run."""
    from xlstm_amd import _lib
    from xlstm_amd import cell as cell_module
    from xlstm_amd.cell import sLSTMCell, sLSTMCellConfig

    print("case stack", native, dtype, dh, flush=True)
    if not native:
        monkeypatch.setattr(cell_module.sLSTMCell_hip, "_trains_natively", lambda self, input: False)
    host, F, H, B, T = _lib.host(), cell_module.F_hip, 2 * dh, 4, 400 if dh == 256 else 8
    torch.manual_seed(dh)
    cells = [sLSTMCell(sLSTMCellConfig(hidden_size=H, num_heads=2, backend="hip", recurrent_weight_init="standard",
                                       output_shape="BSH")).to(DEV) for _ in range(4)]
    x0 = torch.randn(B, T, 4 * H, device=DEV, dtype=dtype)
    leaves = [p for cell in cells for p in cell.parameters()]

    def run():
        x, held = x0, []
        for cell in cells:
            out, _ = cell(x)
            x = x0 + out.repeat(1, 1, 4)
            held.append(host.kept(0))
        return x, held

    assert host.kept(0) == 0
    x, held = run()
    each = held[0]
    assert 0 < each <= 36 * B * T * H and held == [each, 2 * each, 3 * each, 4 * each]
    want = torch.autograd.grad(x.float().square().mean(), leaves)
    assert host.kept(0) == 0  # (the graph's outputs are still there, what it saved is not)
    monkeypatch.setattr(F, "KEPT_COEFFICIENT_BYTES_PER_DEVICE", 2 * each + each // 2)
    x, held = run()
    assert held == [each, 2 * each, 2 * each, 2 * each]
    got = torch.autograd.grad(x.float().square().mean(), leaves, retain_graph=True)
    assert host.kept(0) == (2 * each if dh != 256 else 0)  # (a graph that is kept keeps them, but for the row tiles of 4 rows)
    del x
    assert host.kept(0) == 0
    for a, b in zip(want, got):
        # (other row tiles sum in another order; bfloat16 deltas round once, 2^-8, and so do the gradients between layers)
        tol = (1e-4 if dtype == torch.float32 else 3e-2) * float(a.abs().max())
        torch.testing.assert_close(a, b, rtol=0, atol=tol)


def _contiguous(t):
    return t.clone(memory_format=torch.contiguous_format)


def _misaligned(t):
    return torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)


def _other_order(t):
    return t if t.dim() < 2 else t.transpose(0, -1).contiguous().transpose(0, -1)


@pytest.mark.parametrize("kind,dtype,repack", [
    (k, t, r) for k in ("BNSH", "BSH", "SBNH", "general", "layer") for t in (torch.float32, torch.bfloat16) for r in (_contiguous, _misaligned, _other_order)
    if not (k == "general" and r is _misaligned)  # (the entry points called from Python refuse misaligned tensors with an error)
    and not (k == "layer" and t == torch.bfloat16)])
def test_hooks_may_hand_back_other_layouts(monkeypatch, kind, dtype, repack):
    """What hooks on saved tensors return has the values that were packed, in any memory layout (``save_on_cpu(pin_memory=True)``:
    contiguous in the order of the dimensions)."""
    from xlstm_amd import cell as cell_module
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case saved layouts", kind, dtype, repack.__name__, flush=True)
    if kind == "general":
        monkeypatch.setattr(cell_module.sLSTMCell_hip, "_trains_natively", lambda self, input: False)
    torch.manual_seed(1)
    NH, dh, B, T = 2, 128, 3, 5
    H = NH * dh
    s0 = torch.randn(4, B, H, device=DEV)
    s0[2] = s0[2].abs() + 1.0
    if kind == "layer":
        module = sLSTMLayer(sLSTMLayerConfig(embedding_dim=H, num_heads=NH, backend="hip", recurrent_weight_init="standard")).to(DEV).to(dtype)
        module._norm = lambda y, B, S: y.transpose(1, 2).reshape(B, S, -1)  # (PyTorch's own reads what it saved as dense)
        call = lambda: module(x, slstm_state=s0)
    else:
        module = cell_module.sLSTMCell(cell_module.sLSTMCellConfig(hidden_size=H, num_heads=NH, backend="hip", recurrent_weight_init="standard",
                                                                   output_shape="BNSH" if kind == "general" else kind)).to(DEV)
        call = lambda: module(x, s0)[0]
    x = torch.randn(B, T, H if kind == "layer" else 4 * H, device=DEV).to(dtype).requires_grad_(True)
    leaves = [x, *(p for n, p in module.named_parameters() if n != "group_norm.weight")]
    out = call()
    d = torch.randn_like(out)
    want = torch.autograd.grad(out, leaves, d)
    with torch.autograd.graph.saved_tensors_hooks(repack, lambda t: t):
        out = call()
    got = torch.autograd.grad(out, leaves, d)
    for a, b in zip(want, got):
        # (the same kernels on the same values; sums over 15 tokens by float atomics)
        tol = 2.0 ** -7 if a.dtype == torch.bfloat16 else 1e-5
        torch.testing.assert_close(a, b, rtol=tol, atol=tol * float(a.abs().max()))
