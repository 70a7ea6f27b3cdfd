"""The kernels around the cell of a float32 layer against the same formulas in float64 on the CPU (gradients: autograd
through them); a layer's training call through them against the layer's modules one by one."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from tests._util import geometric_reset_mask

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _close(got, want, what, terms):
    """Sums of ``terms`` float32 products: 2^-24 a term at worst, its square root in earnest; an eighth of the former here."""
    got, want = got.double().cpu(), want.detach()
    assert got.shape == want.shape, what
    err = float((got - want).norm() / want.norm().clamp_min(1e-30))
    bound = 2.0 ** -24 * (8 + terms / 8)
    assert err <= bound, (what, err, bound)


def _front64(x, conv_w, conv_b, gates, reset, state):
    B, T, D = x.shape
    K, NH = conv_w.shape[1], gates[0].shape[0]
    before = torch.zeros(B, K - 1, D, dtype=x.dtype) if state is None else state
    x_all = torch.cat([before, x], 1)
    alive = torch.ones(B, T, dtype=torch.bool)
    pre = conv_b.expand(B, T, D) if conv_b is not None else torch.zeros(B, T, D, dtype=x.dtype)
    for back in range(K):
        if back and reset is not None:  # a document that starts in (t - back, t] cuts the tap off
            start = torch.zeros(B, T, dtype=torch.bool)
            start[:, back - 1:] = reset[:, :T - back + 1] if back <= T else start[:, back - 1:]
            alive = alive & ~start
        pre = pre + torch.where(alive[..., None], x_all[:, K - 1 - back:K - 1 - back + T], 0.0) * conv_w[:, K - 1 - back]
    xc = F.silu(pre)
    heads = [t.view(B, T, NH, D // NH) for t in (xc, xc, x, x)]
    return xc, torch.cat([torch.matmul(h.permute(2, 0, 1, 3).reshape(NH, B * T, -1), w.transpose(1, 2)).permute(1, 0, 2).reshape(B, T, D)
                          for h, w in zip(heads, gates)], -1)


def _norm64(h, w, eps, NH):
    T, B, D = h.shape
    out = F.group_norm(h.transpose(0, 1).reshape(B * T, D), NH, None if w is None else 1.0 + w, None, eps)
    return out.view(B, T, D)


@pytest.mark.parametrize("B,T,NH,dh,K,masked,bias,strided", [
    (1, 2, 1, 8, 4, False, True, False),       # the smallest: one run of tokens, one tile, mostly padding
    (3, 5, 3, 4, 3, True, False, True),        # head dim of one piece; token blocks of a workgroup cross rows
    (2, 33, 2, 64, 2, True, True, False),      # whole tiles of units, ragged tokens
    (1, 21, 1, 96, 4, True, True, False),      # a tile and a half
    (5, 13, 2, 136, 4, True, True, True),      # three column tiles, the last of 8 units; 65 tokens: one behind a tile
    (8, 64, 2, 192, 4, False, True, False),    # eight token tiles: dealt out by XCD
    (7, 301, 1, 40, 4, True, False, False),    # sums over tokens in several slices, the last short
    (2, 600, 2, 32, 4, True, True, True),      # as many slices as there may be
    (2, 24, 1, 296, 4, True, True, False),     # group norm: two pieces a lane
    (1, 9, 2, 512, 4, False, True, False),     # the largest head dim
])
def test_kernels_around_the_cell_equal_float64(B, T, NH, dh, K, masked, bias, strided):
    from xlstm_amd import _lib

    print("case layer f32", B, T, NH, dh, K, masked, bias, strided, flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(B * T + dh)
    D, eps = NH * dh, 1e-5

    def rand(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g) * scale).requires_grad_(True)

    x_wide = torch.randn(B, T, 2 * D, generator=g)
    x = x_wide[..., :D].contiguous().requires_grad_(True)
    conv_w, conv_b, gates = rand(D, K, scale=0.5), rand(D) if bias else None, [rand(NH, dh, dh, scale=dh ** -0.5) for _ in range(4)]
    h, norm_w = torch.randn(T, B, D, generator=g), torch.randn(D, generator=g) * 0.2 if bias else None
    state = torch.randn(B, K - 1, D, generator=g) if not masked else None
    reset = torch.from_numpy(geometric_reset_mask(dh, B, T, 4)) if masked else None
    if masked:
        reset[:, 0] = 0
    d_wx = torch.randn(B, T, 4 * D, generator=g)

    def dbl(t):
        return None if t is None else t.detach().double().requires_grad_(True)

    x64, cw64, cb64, g64 = dbl(x), dbl(conv_w), dbl(conv_b), [dbl(w) for w in gates]
    mask64 = None if reset is None else reset != 0

    def dev(t):
        return None if t is None else t.detach().to(DEV)

    xd = x_wide.to(DEV)[..., :D] if strided else dev(x)
    t = {"conv_w": dev(conv_w), "conv_b": dev(conv_b), "norm_w": dev(norm_w), "reset": dev(reset), "conv_state": dev(state),
         "h": dev(h), "d_wx": dev(d_wx)}
    for name, shape in (("x_conv", (B, T, D)), ("wx", (B, T, 4 * D)), ("out", (B, T, D)), ("d_x_conv", (B, T, D)),
                        ("d_x", (B, T, D)), ("d_conv_w", (D, K)), ("d_conv_b", (D,)),
                        ("scratch", (lib.xs_layer_scratch_floats(B, T, NH, dh, K),))):
        t[name] = torch.full(shape, 7.0, device=DEV)
    gd, d_gates = [dev(w) for w in gates], [torch.full((NH, dh, dh), 7.0, device=DEV) for _ in range(4)]
    a = _lib.LayerArgs()
    a.B, a.T, a.NH, a.dh, a.K, a.eps = B, T, NH, dh, K, eps
    a.x, a.x_stride_b, a.x_stride_t = xd.data_ptr(), xd.stride(0), xd.stride(1)
    for name, v in t.items():
        setattr(a, name, None if v is None else v.data_ptr())
    a.reset_stride_b = T
    for i in range(4):
        a.gate_w[i], a.d_gate_w[i] = gd[i].data_ptr(), d_gates[i].data_ptr()
    a.stream = torch.cuda.current_stream().cuda_stream

    def call(fn):
        rc = fn(ctypes.byref(a))
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()

    xc64, wx64 = _front64(x64, cw64, cb64, g64, mask64, None if state is None else state.double())
    call(lib.xs_layer_front)
    _close(t["x_conv"], xc64, "x_conv", K)
    _close(t["wx"], wx64, "wx", dh)
    call(lib.xs_layer_norm)
    _close(t["out"], _norm64(h.double(), None if norm_w is None else norm_w.double(), eps, NH), "out", dh)
    # the gradients (a state in front of the convolution goes with inference)
    if state is not None:
        a.conv_state = None
        xc64, wx64 = _front64(x64, cw64, cb64, g64, mask64, None)
        call(lib.xs_layer_front)
    wx64.backward(d_wx.double())
    call(lib.xs_layer_front_backward)
    _close(t["d_x"], x64.grad, "d_x", 2 * dh)
    # (the convolution's gradients are sums over tokens of what 2 dh products were summed to: both count)
    _close(t["d_conv_w"], cw64.grad, "d_conv_w", 2 * dh + B * T)
    for i in range(4):
        _close(d_gates[i], g64[i].grad, f"d_gate {i}", B * T)
    if bias:
        _close(t["d_conv_b"], cb64.grad, "d_conv_b", 2 * dh + B * T)
    else:
        assert bool((t["d_conv_b"] == 7.0).all())
    # what is not wanted is not made; the rest comes out the same
    results = {"d_x": t["d_x"], "d_conv_w": t["d_conv_w"], "d_conv_b": t["d_conv_b"], **{i: d_gates[i] for i in range(4)}}
    whole = {k: v.clone() for k, v in results.items()}
    for wanted in (("d_x",), ("d_conv_w",), ("d_conv_b",), (0, 3), (2, "d_conv_w"), ("d_x", 1), ()):
        for k, v in [*results.items(), *t.items()]:
            if k in results or k in ("d_x_conv", "scratch"):
                v.fill_(7.0)
            if k in results and isinstance(k, str):
                setattr(a, k, v.data_ptr() if k in wanted else None)
            elif k in results:
                a.d_gate_w[k] = v.data_ptr() if k in wanted else None
        call(lib.xs_layer_front_backward)
        for k, v in results.items():
            made = k in wanted and (k != "d_conv_b" or bias)
            assert torch.equal(v, whole[k]) if made else bool((v == 7.0).all()), (wanted, k)
        if not any(isinstance(k, str) for k in wanted):
            assert bool((t["d_x_conv"] == 7.0).all())


def _layer(NH, dh, **kw):
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    torch.manual_seed(dh)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=NH * dh, num_heads=NH, backend="hip", recurrent_weight_init="standard", **kw)).to(DEV)
    with torch.no_grad():
        layer.group_norm.weight.normal_(0, 0.2)
    return layer


def _one_node(out):
    """Whether the graph behind ``out`` has the node of a layer's training call."""
    todo, seen = [out.grad_fn], set()
    while todo:
        fn = todo.pop()
        if fn is None or fn in seen:
            continue
        if "sLSTMLayer" in fn.name():
            return True
        seen.add(fn)
        todo += [f for f, _ in fn.next_functions]
    return False


def _training_call(layer, x, state, mask, last, d_out, d_state):
    out = layer(x, slstm_state=state, reset_mask=mask, return_last_state=last)
    out, states = out if last else (out, None)
    leaves = [x, *layer.parameters()] + ([state] if state is not None else [])
    heads, grads = [out], [d_out]
    if last:
        heads, grads = heads + [states["slstm_state"], states["conv_state"]], grads + [d_state, torch.ones_like(states["conv_state"])]
    return out, states, leaves, torch.autograd.grad(heads, leaves, grads, retain_graph=True)


@pytest.mark.parametrize("B,T,NH,dh,mask,last,extra", [
    (2, 9, 2, 64, True, False, {}), (3, 4, 1, 96, False, True, dict(state=True)), (1, 30, 4, 128, True, True, {}),
    (4, 5, 2, 48, True, False, dict(expanded=True, transposed=True)), (2, 7, 1, 200, False, False, dict(cut=True, clip=1.0)),
])
def test_training_call_of_a_layer_equals_its_modules_one_by_one(B, T, NH, dh, mask, last, extra):
    print("case layer training", B, T, NH, dh, mask, last, extra, flush=True)
    D = NH * dh
    layer = _layer(NH, dh, gradient_recurrent_cut=bool(extra.get("cut")), gradient_recurrent_clipval=extra.get("clip"))
    x = torch.randn(B, T, D, device=DEV)
    if extra.get("transposed"):
        x = torch.randn(T, B, D, device=DEV).transpose(0, 1)
    x = x.requires_grad_(True)
    state = None
    if extra.get("state"):
        state = torch.randn(4, B, D, device=DEV)
        state[2] = state[2].abs() + 1.0
        state.requires_grad_(True)
    m = torch.from_numpy(geometric_reset_mask(1, B, T, 3)).to(DEV).bool() if mask else None
    d_out = torch.ones(1, device=DEV).expand(B, T, D) if extra.get("expanded") else torch.randn(B, T, D, device=DEV)
    d_state = torch.randn(4, B, D, device=DEV)
    out, states, leaves, got = _training_call(layer, x, state, m, last, d_out, d_state)
    assert _one_node(out)
    layer.fused_pre_ops = False
    ref, ref_states, _, want = _training_call(layer, x, state, m, last, d_out, d_state)
    layer.fused_pre_ops = True
    assert not _one_node(ref)
    # float32 on both sides: sums over dh units, then over up to 30 steps of a recurrence
    torch.testing.assert_close(out, ref, rtol=1e-4, atol=1e-5)
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4 * float(b.detach().abs().max()))
    if last:
        torch.testing.assert_close(states["slstm_state"], ref_states["slstm_state"], rtol=1e-4, atol=1e-5)
        assert torch.equal(states["conv_state"], ref_states["conv_state"])
    # a backward that is recorded itself gives the general path's gradients and graph
    first = torch.autograd.grad(out, leaves, d_out, create_graph=True, allow_unused=True)
    second = torch.autograd.grad(ref, leaves, d_out, create_graph=True, allow_unused=True)
    for a, b in zip(first, second):
        assert (a is None) == (b is None) and (a is None or a.requires_grad == b.requires_grad)
        if a is not None:
            torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4 * float(b.detach().abs().max()))
    with torch.no_grad():  # inference through the same kernels
        quiet = layer(x, slstm_state=state, reset_mask=m)
        layer.fused_pre_ops = False
        torch.testing.assert_close(quiet, layer(x, slstm_state=state, reset_mask=m), rtol=1e-4, atol=1e-5)


def test_inference_continues_from_states():
    print("case layer f32 states", flush=True)
    layer = _layer(2, 40)
    x = torch.randn(3, 17, 80, device=DEV)
    with torch.no_grad():
        whole = layer(x)
        first, st = layer(x[:, :9], return_last_state=True)
        second = layer(x[:, 9:], conv_state=st["conv_state"], slstm_state=st["slstm_state"])
    torch.testing.assert_close(torch.cat([first, second], 1), whole, rtol=1e-5, atol=1e-5)


def test_inputs_off_the_16_bytes_of_the_kernels():
    """x as a contiguous view that starts 4 bytes into an allocation: laid out again, as a view with other strides is."""
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case misaligned", flush=True)
    torch.manual_seed(3)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=96, num_heads=3, backend="hip", recurrent_weight_init="standard")).to(DEV).eval()
    x = torch.randn(2, 9, 96, device=DEV)
    off = torch.empty(x.numel() + 1, device=DEV)[1:].view(x.shape).copy_(x)
    assert off.is_contiguous() and off.data_ptr() % 16
    with torch.no_grad():
        want, states = layer(x, return_last_state=True)
        got, got_states = layer(off, return_last_state=True)
    assert torch.equal(got, want) and torch.equal(got_states["slstm_state"], states["slstm_state"])
    assert torch.equal(got_states["conv_state"], states["conv_state"])


def test_what_wants_the_modules_one_by_one_gets_them():
    print("case layer f32 modules", flush=True)
    layer = _layer(2, 64)
    x = torch.randn(2, 6, 128, device=DEV, requires_grad=True)

    def native():
        return _one_node(layer(x))

    assert native()
    seen = []
    for register in ("register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook"):
        for m in (layer.igate, layer.conv1d, layer.conv1d.conv, layer.conv_act_fn, layer.slstm_cell):
            handle = getattr(m, register)(lambda *_: seen.append(1) and None)
            assert not native(), (register, m)
            handle.remove()
    seen.clear()
    for m in (layer.group_norm, layer.dropout):  # (called in a training call too; inference leaves its path for them)
        handle = m.register_forward_hook(lambda *_: seen.append(1) and None)
        assert native()
        with torch.no_grad():
            layer(x)
        handle.remove()
    assert len(seen) == 4
    assert native()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not native()
    layer.dropout.p = 0.5
    a, b = layer(x), layer(x)
    assert _one_node(a) and not torch.equal(a, b)
    layer.dropout.p = 0.0
    weight = layer.igate.weight
    del layer.igate.weight  # a weight that is made from another tensor
    layer.igate.weight = weight * 1.0
    assert not native()
    del layer.igate.weight
    layer.igate.weight = weight
    assert native()
    inner = layer.zgate
    layer.zgate = torch.nn.Sequential(inner)
    assert not native()
    layer.zgate = inner
    out = layer(x)
    with torch.no_grad():
        layer.conv1d.conv.weight.mul_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()
    out = layer(x)
    out.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        out.sum().backward()


@pytest.mark.parametrize("chain", ["state", "input", "tied"])
def test_recorded_backward_of_calls_that_depend_on_the_layer(chain):
    """A backward pass that is itself recorded, where x or the state of a call comes from an earlier call of the same layer, or one weight
    serves two gates: every call's share is counted once."""
    print("case layer create_graph", chain, flush=True)
    layer = _layer(2, 64)
    if chain == "tied":
        layer.zgate.weight = layer.ogate.weight
    x0, x1 = (torch.randn(2, 6, 128, device=DEV, requires_grad=True) for _ in range(2))
    d = torch.randn(2, 6, 128, device=DEV)

    def gradients(fused, create_graph):
        layer.fused_pre_ops = fused
        first, states = layer(x0, return_last_state=True)
        out = layer(first) if chain == "input" else layer(x1, slstm_state=states["slstm_state"])
        assert _one_node(out) is fused
        leaves = [x0, x1, *layer.parameters()]
        return torch.autograd.grad([first, out], leaves, [d, d], create_graph=create_graph, allow_unused=True)

    want = gradients(False, False)
    for got in (gradients(True, True), gradients(True, False)):
        for a, b in zip(got, want):
            assert (a is None) == (b is None)
            if a is not None:  # (float32 on both sides: sums over dh units, then over 12 steps of a recurrence)
                torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4 * float(b.detach().abs().max()))


def test_recorded_backward_leaves_the_layers_parameters_in_place(monkeypatch):
    """Other threads may be in the layer while a recorded backward makes a call's operations once more."""
    from xlstm_amd import layer as layer_module

    print("case layer create_graph in place", flush=True)
    layer = _layer(2, 64)
    mine = dict(layer.named_parameters())
    x = torch.randn(2, 6, 128, device=DEV, requires_grad=True)
    out = layer(x)
    assert _one_node(out)
    forward, seen = layer_module.CausalConv1d.forward, []

    def watched(self, *args, **kwargs):
        now = dict(layer.named_parameters())
        seen.append(self is not layer.conv1d and set(now) == set(mine) and all(now[n] is mine[n] for n in mine))
        return forward(self, *args, **kwargs)

    monkeypatch.setattr(layer_module.CausalConv1d, "forward", watched)
    grads = torch.autograd.grad(out, [x, *mine.values()], torch.ones_like(out), create_graph=True)
    assert seen == [True] and all(g.isfinite().all() for g in grads)
    layer.slstm_cell.check_status()


def test_what_a_training_call_returned_does_not_hold_the_layer():
    """An output kept on the layer goes with it, and its graph outlives the layer."""
    import gc
    import weakref

    print("case layer kept output", flush=True)
    layer = _layer(2, 64)
    x = torch.randn(2, 6, 128, device=DEV, requires_grad=True)
    out = layer(x)
    assert _one_node(out)
    layer.last, gone = layer(x), weakref.ref(layer)
    leaves = [x, *layer.parameters()]
    want = torch.autograd.grad(layer(x), leaves, torch.ones_like(out))
    kept = weakref.ref(layer.last)
    del layer
    gc.collect()
    assert gone() is None and kept() is None
    got = torch.autograd.grad(out, leaves, torch.ones_like(out), create_graph=True)
    for a, b in zip(got, want):  # (float32 on both sides: sums over dh units, then over 6 steps of a recurrence)
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4 * float(b.abs().max()))


@pytest.mark.parametrize("frozen", [("x",), ("fgate", "igate", "zgate", "ogate"), ("conv1d", "x"), ("zgate", "conv1d"), ("conv1d", "fgate", "igate", "zgate", "ogate", "x")])
def test_frozen_parts_of_a_layer(frozen):
    """The gradients of what is not frozen, and of what a call of torch.autograd.grad asks for, are those of the whole."""
    print("case layer frozen", frozen, flush=True)
    layer = _layer(2, 64)
    x = torch.randn(3, 90, 128, device=DEV, requires_grad=True)
    d = torch.randn(3, 90, 128, device=DEV)
    named = {"x": x, **dict(layer.named_parameters())}
    out = layer(x)
    assert _one_node(out)
    whole = dict(zip(named, torch.autograd.grad(out, list(named.values()), d, retain_graph=True)))
    wanted = [n for n in named if n.split(".")[0] not in frozen]
    asked = torch.autograd.grad(out, [named[n] for n in wanted], d)
    for n in named:
        named[n].requires_grad_(n in wanted)
    out = layer(x)
    assert _one_node(out)
    out.backward(d)
    for n, got in zip(wanted, asked):
        # (R and bias are summed by float atomics; the rest has a fixed order)
        tol = 1e-5 * float(whole[n].abs().max()) if "slstm_cell" in n else 0.0
        torch.testing.assert_close(got, whole[n], rtol=0, atol=tol)
        torch.testing.assert_close(named[n].grad, whole[n], rtol=0, atol=tol)
    assert all(named[n].grad is None for n in named if n not in wanted)


@pytest.mark.parametrize("own", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S", [(1, 3), (4, 32), (3, 43), (8, 512)])
def test_gradients_of_the_norm(B, S, dtype, own):
    """A group norm's gradients against float64 on the CPU.  That of the weight is PyTorch's up to 128 tokens and wrong there beyond, of
    which the call warns; with own_weight_gradient it is right at any number of them."""
    import warnings

    from xlstm_amd import layer as layer_module

    print("case norm gradients", B, S, dtype, own, flush=True)
    NH, dh = 2, 64
    torch.manual_seed(B * S)
    norm = layer_module.MultiHeadLayerNorm(NH * dh).to(DEV).to(dtype)
    with torch.no_grad():
        norm.weight.normal_(std=0.2)
    norm.own_weight_gradient = own
    y = torch.randn(S, B, NH, dh, device=DEV).to(dtype).permute(1, 2, 0, 3).requires_grad_(True)
    d = torch.randn(B, NH, S, dh, device=DEV).to(dtype)
    layer_module._warn_of_the_weight_gradient.cache_clear()
    with warnings.catch_warnings(record=True) as said:
        warnings.simplefilter("always")
        for _ in range(2):
            out = norm(y)
        with torch.no_grad():
            assert torch.equal(norm(y), out)  # (the same bits, whatever makes the gradient)
    wrong = B * S > 128 and not own
    assert sum("group norm" in str(w.message) for w in said) == wrong  # (once)
    got = torch.autograd.grad(out, (y, norm.weight), d)
    y64 = y.detach().double().cpu().requires_grad_(True)
    scale = 1.0 + norm.weight.detach().cpu()  # (rounded to the module's type, as the module does)
    w64 = scale.double().requires_grad_(True)
    want64 = _norm64(y64.permute(2, 0, 1, 3).reshape(S, B, NH * dh), w64 - 1.0, norm.eps, NH).reshape(B, S, NH, dh).transpose(1, 2)
    want = torch.autograd.grad(want64, (y64, w64), d.double().cpu())
    # float32: a few sums of 64 products, then over 4096 tokens, whose rounding errors grow with the square root: 2^-24 times 8 + 64.
    # bfloat16: results of float32 sums, rounded once
    bound = 2.0 ** -24 * 72 if dtype == torch.float32 else 2.0 ** -8
    for a, b in list(zip(got, want))[: 1 if wrong else 2]:
        assert float((a.double().cpu() - b).norm() / b.norm()) <= bound
