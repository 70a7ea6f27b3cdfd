"""The two HIP kernels in front of the cell (convolution + SiLU, headwise gate projections) against float32
PyTorch restatements of the same operations on the same bf16-rounded operands.  Tolerance 2e-2 on
max |a - d| / max(1, |d|), the bf16 bar of the cell; the outputs are float32 results rounded once to bf16."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from tests._util import geometric_reset_mask, max_err

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = 2e-2


def conv_silu_reference(x, w, bias, conv_state, mask):
    """float32, per document: silu(causal depthwise conv) with taps cut at document starts."""
    B, T, D = x.shape
    K = w.shape[1]
    x = x.float(); w = w.float()
    prev = torch.zeros(B, K - 1, D) if conv_state is None else conv_state.float()
    xa = torch.cat([prev, x], 1)  # token t sits at t + K - 1
    out = torch.zeros(B, T, D)
    for b in range(B):
        last_start = None
        for t in range(T):
            if mask is not None and mask[b, t]:
                last_start = t
            acc = torch.zeros(D) if bias is None else bias.float().clone()
            for back in range(K):
                ts = t - back
                if last_start is not None and ts < last_start:
                    continue
                acc = acc + w[:, K - 1 - back] * xa[b, ts + K - 1]
            out[b, t] = acc
    return F.silu(out)


@pytest.mark.parametrize("B,T,D,K,with_state,with_mask,with_bias", [
    (2, 19, 64, 4, False, False, True),
    (3, 33, 128, 4, True, True, True),
    (1, 7, 8, 3, True, False, False),
    (2, 40, 24, 2, False, True, True),
    (5, 1, 256, 4, True, False, True),  # a decode step
])
def test_causal_conv_silu_equals_float32_restatement(B, T, D, K, with_state, with_mask, with_bias):
    from xlstm_amd import functional as hipF

    g = torch.Generator().manual_seed(B * 1000 + T)
    x = torch.randn(B, T, D, generator=g).bfloat16()
    w = (torch.randn(D, K, generator=g) * 0.5).bfloat16()
    bias = torch.randn(D, generator=g).bfloat16() if with_bias else None
    state = torch.randn(B, K - 1, D, generator=g).bfloat16() if with_state else None
    mask = None
    if with_mask:
        mask = torch.from_numpy(geometric_reset_mask(T, B, T, 5))
        mask[:, 0] = 0  # the first document continues from conv_state / zero padding
        mask[0, 1] = 1; mask[0, 2] = 1  # documents of one token
    want = conv_silu_reference(x, w, bias, state, mask)
    got = hipF.causal_conv_silu(x.to(DEV), w.view(D, 1, K).to(DEV), None if bias is None else bias.to(DEV),
                                None if state is None else state.to(DEV), None if mask is None else mask.to(DEV))
    torch.cuda.synchronize()
    assert got.dtype == torch.bfloat16 and tuple(got.shape) == (B, T, D)
    assert max_err(got.float().cpu().numpy(), want.numpy()) <= TOL


def test_causal_conv_silu_reads_a_ring_view_and_strided_input():
    """conv_state as the [:, :-1] view of a [B,K,D] ring and x as a slice of a longer sequence: no copies needed."""
    from xlstm_amd import functional as hipF

    g = torch.Generator().manual_seed(5)
    B, D, K = 4, 128, 4
    ring = torch.randn(B, K, D, generator=g).bfloat16()
    w = torch.randn(D, K, generator=g).bfloat16()
    bias = torch.randn(D, generator=g).bfloat16()
    x = ring[:, -1:]
    want = conv_silu_reference(x, w, bias, ring[:, :-1], None)
    ring_d = ring.to(DEV)
    got = hipF.causal_conv_silu(ring_d[:, -1:], w.to(DEV), bias.to(DEV), ring_d[:, :-1])
    assert max_err(got.float().cpu().numpy(), want.numpy()) <= TOL
    long = torch.randn(B, 30, D, generator=g).bfloat16()
    want = conv_silu_reference(long[:, 10:25], w, bias, long[:, 7:10], None)
    long_d = long.to(DEV)
    got = hipF.causal_conv_silu(long_d[:, 10:25], w.to(DEV), bias.to(DEV), long_d[:, 7:10])
    assert max_err(got.float().cpu().numpy(), want.numpy()) <= TOL


def test_causal_conv_silu_step_writes_the_next_ring():
    from xlstm_amd import functional as hipF

    g = torch.Generator().manual_seed(6)
    B, D, K = 3, 64, 4
    ring = torch.randn(B, K, D, generator=g).bfloat16().to(DEV)
    x = torch.randn(B, 1, D, generator=g).bfloat16().to(DEV)
    w = torch.randn(D, K, generator=g).bfloat16().to(DEV)
    new_ring = torch.full((B, K, D), 7.0, dtype=torch.bfloat16, device=DEV)
    got = hipF.causal_conv_silu(x, w, None, ring[:, 1:], ring_out=new_ring)
    want = hipF.causal_conv_silu(x, w, None, ring[:, 1:].contiguous())
    assert torch.equal(got, want)
    assert torch.equal(new_ring, torch.cat([ring[:, 1:], x], 1))
    first = torch.full((B, K, D), 7.0, dtype=torch.bfloat16, device=DEV)  # no state yet: zeros, then x
    hipF.causal_conv_silu(x, w, None, None, ring_out=first)
    assert torch.equal(first, torch.cat([torch.zeros(B, K - 1, D, dtype=torch.bfloat16, device=DEV), x], 1))
    with pytest.raises(hipF.EngineError):
        hipF.causal_conv_silu(x, w, None, ring[:, 1:], ring_out=ring)  # in place is refused


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("dtype,NH,dh,K", [(torch.float32, 3, 40, 4), (torch.float32, 2, 64, 2), (torch.bfloat16, 2, 64, 4), (torch.bfloat16, 1, 128, 3)])
def test_one_convolution_state_for_all_rows(dtype, NH, dh, K, native, monkeypatch):
    """A state expanded over the batch (rows of stride 0): the same as its copies, in sequences and in steps, through the native host path
    and the kernels of the parts.  (float32: such a call takes PyTorch's operations around the cell, whose sums round in another order.)"""
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case shared conv state", dtype, NH, dh, K, native, flush=True)
    torch.manual_seed(K)
    B, D = 5, NH * dh
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=D, num_heads=NH, conv1d_kernel_size=K, backend="hip", recurrent_weight_init="standard")).to(DEV, dtype).eval()
    layer.slstm_cell.keep_state_fp32 = True
    if not native:
        monkeypatch.setattr(layer, "_own_modules", lambda: False)
    x = torch.randn(B, 6, D, device=DEV).to(dtype)
    token = torch.randn(B, 1, D, device=DEV).to(dtype)
    rows = [torch.randn(1, n, D, device=DEV).to(dtype).expand(B, n, D) for n in (K - 1, K)]
    overlapping = torch.randn((B + K) * D, device=DEV).to(dtype).as_strided((B, K - 1, D), (max(D // 8 * 8, 8), D, 1))
    tolerance = dict(rtol=1e-5, atol=1e-5) if dtype == torch.float32 else dict(rtol=0, atol=0)
    with torch.no_grad():
        state = layer(x, return_last_state=True)[1]["slstm_state"].float()
        for taps in (*rows, overlapping):
            torch.testing.assert_close(layer(x, conv_state=taps), layer(x, conv_state=taps.contiguous()), **tolerance)
            for _ in range(2):  # (the second on the plan of the first)
                got, want = (layer.step(token, conv_state=(t,), slstm_state=state) for t in (taps, taps.contiguous()))
                torch.testing.assert_close(got[0], want[0], **tolerance)
                assert torch.equal(got[1]["conv_state"][0], want[1]["conv_state"][0])


@pytest.mark.parametrize("B,D,K", [(1, 8, 2), (3, 64, 3), (37, 520, 4)])
def test_a_token_is_left_in_another_buffer_too(B, D, K):
    import ctypes

    from xlstm_amd import _lib
    from xlstm_amd import functional as hipF

    print("case token out", B, D, K, flush=True)
    torch.manual_seed(B)
    memory = torch.randn(8 * B * K, D, device=DEV).bfloat16()  # (one allocation: what overlaps is known)
    x, taps, out, ring, free = (memory[i * B * K:(i + 1) * B * K] for i in range(5))
    w = torch.randn(D, K, device=DEV).bfloat16()
    a = _lib.ConvArgs()
    a.B, a.T, a.D, a.K, a.dtype = B, 1, D, K, _lib.XS_BF16
    a.x, a.x_stride_b, a.x_stride_t, a.conv_state, a.weight, a.out = x.data_ptr(), D, D, taps.data_ptr(), w.data_ptr(), out.data_ptr()
    a.stream = torch.cuda.current_stream().cuda_stream
    call = _lib.load().xs_causal_conv_silu_token
    assert call(ctypes.byref(a), free.data_ptr()) == -1  # goes with a ring
    a.ring_out = ring.data_ptr()
    assert call(ctypes.byref(a), None) == -1 and call(ctypes.byref(a), free.data_ptr() + 2) == -4
    before = memory.clone()
    last = {"x": x[B - 1:], "conv_state": taps[B * (K - 1) - 1:], "out": out[B - 1:], "ring_out": ring[B * K - 1:]}
    for name, rows in last.items():
        assert call(ctypes.byref(a), rows.data_ptr()) == -2 and name.encode() in _lib.load().xs_last_error(), name
    torch.cuda.synchronize()
    assert torch.equal(memory, before)
    assert call(ctypes.byref(a), free.data_ptr()) == 0
    torch.cuda.synchronize()
    states = taps[:B * (K - 1)].view(B, K - 1, D)
    want = hipF.causal_conv_silu(x[:B].view(B, 1, D), w, None, states)
    assert torch.equal(free[:B], x[:B]) and torch.equal(free[B:], before[4 * B * K + B:5 * B * K])
    assert torch.equal(out[:B], want[:, 0]) and torch.equal(ring.view(B, K, D), torch.cat([states, x[:B].view(B, 1, D)], 1))


@pytest.mark.parametrize("lead,NH,dh", [
    ((2, 37), 4, 64),      # 64-token x 64-unit tiles, ragged token count
    ((3, 50), 2, 256),     # 64 x 128
    ((4, 1100), 4, 128),   # 128 x 128 (>= 4096 tokens), ragged
    ((4100,), 4, 64),      # 128 x 64, ragged
    ((256, 1), 8, 256),    # the decode shape of BASELINE config 3
    ((1, 1), 1, 192),      # one token, three 64-unit tiles per slot
    ((8, 2048), 4, 256),   # the layer of BASELINE config 4: weights resident, 8 token partitions of 16 tiles
    ((5, 999), 16, 256),   # 128 combinations: two token partitions, no XCD grouping, ragged
    ((3, 1000), 3, 128),   # 12 combinations, 16 partitions of one or two tiles
    ((2, 3), 1, 128),      # fewer token tiles than partitions
])
def test_headwise_gates_equal_float32_einsum(lead, NH, dh):
    from xlstm_amd import functional as hipF

    g = torch.Generator().manual_seed(NH * dh + len(lead))
    H = NH * dh
    x = torch.randn(*lead, H, generator=g).bfloat16()
    xc = torch.randn(*lead, H, generator=g).bfloat16()
    ws = [(torch.randn(NH, dh, dh, generator=g) / np.sqrt(dh)).bfloat16() for _ in range(4)]
    want = torch.cat([torch.einsum("...hd,hod->...ho", (xc if s < 2 else x).float().view(*lead, NH, dh), ws[s].float()).reshape(*lead, H)
                      for s in range(4)], dim=-1)
    got = hipF.headwise_gates(x.to(DEV), xc.to(DEV), [w.to(DEV) for w in ws], NH)
    torch.cuda.synchronize()
    assert got.dtype == torch.bfloat16 and tuple(got.shape) == tuple(lead) + (4 * H,)
    assert max_err(got.float().cpu().numpy(), want.numpy()) <= TOL


def test_headwise_gates_slot_wiring_one_hot():
    """Exact check of the indexing: with one-hot operands every output is a single weight, bit for bit."""
    from xlstm_amd import functional as hipF

    NH, dh = 2, 64
    H = NH * dh
    g = torch.Generator().manual_seed(9)
    ws = [torch.randn(NH, dh, dh, generator=g).bfloat16() for _ in range(4)]
    x = torch.zeros(3, H).bfloat16(); xc = torch.zeros(3, H).bfloat16()
    x[0, 5] = 1; x[1, 64 + 17] = 1; x[2, 63] = 1        # z, o read x
    xc[0, 64 + 3] = 1; xc[1, 9] = 1; xc[2, 127] = 1     # i, f read x_conv
    got = hipF.headwise_gates(x.to(DEV), xc.to(DEV), [w.to(DEV) for w in ws], NH).cpu()
    for m, (cx, cxc) in enumerate([(5, 64 + 3), (64 + 17, 9), (63, 127)]):
        for s in range(4):
            c = cxc if s < 2 else cx
            h, d = divmod(c, dh)
            want = torch.zeros(H).bfloat16()
            want[h * dh:(h + 1) * dh] = ws[s][h, :, d]
            assert torch.equal(got[m, s * H:(s + 1) * H], want), (m, s)


@pytest.mark.parametrize("B,NH,T,dh,with_weight,cell_layout", [
    (3, 4, 17, 64, True, True),
    (2, 2, 5, 256, True, True),
    (2, 3, 9, 36, False, False),    # 9 pieces of 4 units: part of a wave idles
    (1, 1, 4, 1024, True, True),    # four pieces per lane
    (5, 2, 1, 520, True, False),    # three pieces used of four
])
def test_headwise_group_norm_equals_float32_group_norm(B, NH, T, dh, with_weight, cell_layout):
    from xlstm_amd import functional as hipF

    g = torch.Generator().manual_seed(B + NH + T + dh)
    H = NH * dh
    if cell_layout:  # the cell's output: [S,B,H] storage seen as [B,NH,S,DH] (cell.py:354-374)
        y = (torch.randn(T, B, H, generator=g) * 3 + 0.5).bfloat16().view(T, B, NH, dh).permute(1, 2, 0, 3)
    else:
        y = (torch.randn(B, NH, T, dh, generator=g) * 3 + 0.5).bfloat16()
    w = (torch.randn(H, generator=g) * 0.2).bfloat16() if with_weight else None
    want = F.group_norm(y.float().transpose(1, 2).reshape(B * T, H), NH, None if w is None else 1.0 + w.float(), None, 1e-5)
    got = hipF.headwise_group_norm(y.to(DEV), None if w is None else w.to(DEV), 1e-5)
    torch.cuda.synchronize()
    assert got.dtype == torch.bfloat16 and tuple(got.shape) == (B, T, H)
    assert max_err(got.float().cpu().numpy(), want.view(B, T, H).numpy()) <= TOL


def test_layer_with_engine_pre_ops_equals_layer_with_torch_pre_ops():
    """sLSTMLayer.forward and .step: the HIP conv / projection kernels against the PyTorch ops they replace."""
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    torch.manual_seed(11)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=256, num_heads=4, backend="hip",
                                        recurrent_weight_init="standard")).to(DEV).bfloat16().eval()
    layer.slstm_cell.keep_state_fp32 = True
    x = torch.randn(3, 40, 256, device=DEV).bfloat16()
    mask = torch.from_numpy(geometric_reset_mask(2, 3, 40, 9)).to(DEV)
    with torch.no_grad():
        assert layer._fused(x)
        fused, st_f = layer(x, reset_mask=mask, return_last_state=True)
        o_f, st_f2 = layer.step(x[:, :1], conv_state=st_f["conv_state"], slstm_state=st_f["slstm_state"])
        layer.fused_pre_ops = False
        plain, st_p = layer(x, reset_mask=mask, return_last_state=True)
        o_p, st_p2 = layer.step(x[:, :1], conv_state=st_p["conv_state"], slstm_state=st_p["slstm_state"])
        # a forward continues from the ring a step returned (k inputs) and from a shorter state alike
        layer.fused_pre_ops = True
        a1 = layer(x[:, 1:9], conv_state=st_f2["conv_state"])
        a2 = layer(x[:, 1:9], conv_state=st_f2["conv_state"][0][:, -2:])
        layer.fused_pre_ops = False
        b1 = layer(x[:, 1:9], conv_state=st_p2["conv_state"])
        b2 = layer(x[:, 1:9], conv_state=st_p2["conv_state"][0][:, -2:])
        # the same layer in float32 (bf16-rounded parameters, PyTorch ops, float32 cell kernel): the yardstick
        import copy

        ref_layer = copy.deepcopy(layer).float()
        ref_layer.fused_pre_ops = False
        ref32 = ref_layer(x.float(), reset_mask=mask)
    # The engine's layer path against the float32 layer at the bf16 bar.  The PyTorch bf16 path rounds after every op
    # (conv, SiLU, each projection) and is itself up to that far from float32, so the two bf16 pipelines are compared
    # with each other at the sum of the two bars, after the group norm has divided by a head's spread.
    e_fused = max_err(fused.float().cpu().numpy(), ref32.cpu().numpy())
    e_plain = max_err(plain.float().cpu().numpy(), ref32.cpu().numpy())
    print("layer vs float32 layer: engine ops %.3e, torch ops %.3e" % (e_fused, e_plain), flush=True)
    assert e_fused <= 2e-2
    assert max_err(fused.float().cpu().numpy(), plain.float().cpu().numpy()) <= 2e-2 + max(e_plain, 2e-2)
    assert max_err(a1.float().cpu().numpy(), b1.float().cpu().numpy()) <= 5e-2
    assert max_err(a2.float().cpu().numpy(), b2.float().cpu().numpy()) <= 5e-2
    assert torch.equal(st_f["conv_state"], st_p["conv_state"])
    assert max_err(st_f["slstm_state"].cpu().numpy(), st_p["slstm_state"].cpu().numpy()) <= 5e-2
    assert max_err(o_f.float().cpu().numpy(), o_p.float().cpu().numpy()) <= 5e-2
    assert torch.equal(st_f2["conv_state"][0], st_p2["conv_state"][0])


def test_layer_under_autograd_keeps_the_pytorch_ops_and_trains_through_the_cell():
    """The engine's layer kernels record no graph: with grad enabled the layer keeps its PyTorch ops around the cell,
    and the cell's own backward kernels carry the gradient (head dims in between their sizes run padded)."""
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    torch.manual_seed(12)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=256, num_heads=4, backend="hip")).to(DEV).bfloat16()
    x = torch.randn(2, 6, 256, device=DEV).bfloat16().requires_grad_(True)
    with torch.no_grad():
        assert layer._fused(x)
    assert not layer._fused(x)  # parameters require grad and grad mode is on
    out = layer(x)
    assert out.requires_grad
    out.float().sum().backward()
    grads = [p.grad for p in layer.parameters()]
    assert all(g is not None and torch.isfinite(g.float()).all() for g in grads)
    assert x.grad is not None and torch.isfinite(x.grad.float()).all() and x.grad.float().abs().max() > 0
    small = sLSTMLayer(sLSTMLayerConfig(embedding_dim=256, num_heads=8, backend="hip")).to(DEV).bfloat16()  # head dim 32: padded
    small(x.detach()).float().sum().backward()
    assert all(p.grad is not None and torch.isfinite(p.grad.float()).all() for p in small.parameters())


def test_layer_ops_accept_empty_inputs():
    from xlstm_amd import functional as hipF

    w = torch.zeros(64, 4, dtype=torch.bfloat16, device=DEV)
    assert tuple(hipF.causal_conv_silu(torch.zeros(2, 0, 64, dtype=torch.bfloat16, device=DEV), w).shape) == (2, 0, 64)
    assert tuple(hipF.causal_conv_silu(torch.zeros(0, 5, 64, dtype=torch.bfloat16, device=DEV), w).shape) == (0, 5, 64)
    ws = [torch.zeros(1, 64, 64, dtype=torch.bfloat16, device=DEV)] * 4
    e = torch.zeros(0, 3, 64, dtype=torch.bfloat16, device=DEV)
    assert tuple(hipF.headwise_gates(e, e, ws, 1).shape) == (0, 3, 256)
    assert tuple(hipF.headwise_group_norm(torch.zeros(2, 1, 0, 64, dtype=torch.bfloat16, device=DEV)).shape) == (2, 0, 64)
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 2, 7])
def test_gradient_of_the_inputs_before_x(dtype, T):
    """A layer whose parameters are frozen: the convolution's state and the cell's may still want their gradients."""
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case conv_state gradient", dtype, T, flush=True)
    torch.manual_seed(T)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=128, num_heads=2, backend="hip", recurrent_weight_init="standard")).to(DEV).to(dtype)
    layer.requires_grad_(False)
    x = torch.randn(3, T, 128, device=DEV).to(dtype)
    before = torch.randn(3, 3, 128, device=DEV).to(dtype).requires_grad_(True)
    state = (torch.rand(4, 3, 128, device=DEV) + 0.5).to(dtype).requires_grad_(True)
    d = torch.randn(3, T, 128, device=DEV).to(dtype)
    buffer = torch.empty(3, 1, 128, device=DEV, dtype=dtype)
    with torch.no_grad():  # (plans steps of 3 rows, so that the native host path is asked)
        layer.step(x[:, :1].contiguous(), (before,), state.float())

    def call(wanted):
        ring, s = (t if any(t is w for w in wanted) else t.detach() for t in (before, state))
        return layer.step(x, (ring,), s.float(), out=buffer)[0] if T == 1 else layer(x, conv_state=ring, slstm_state=s)

    for wanted in ((before,), (state,), (before, state)):
        got = torch.autograd.grad(call(wanted), wanted, d)
        layer.fused_pre_ops = False
        want = torch.autograd.grad(call(wanted), wanted, d)
        layer.fused_pre_ops = True
        for a, b in zip(got, want):
            assert a.shape == b.shape and float(b.float().norm()) > 0
            # Where the state alone wants one, the engine's kernels run in front of the cell on one side and PyTorch's on the other.  bfloat16:
            # each of about ten operations rounds to 8 bits, 2^-9 each at worst; float32: sums of 64 products, 2^-24 a term
            bound = 10 * 2.0 ** -9 if dtype == torch.bfloat16 else 10 * 64 * 2.0 ** -24
            assert float((a.float() - b.float()).norm() / b.float().norm()) <= bound


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_norm_without_weights_takes_the_native_host_path(dtype):
    from xlstm_amd import _lib
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case norm without weights", dtype, flush=True)
    torch.manual_seed(0)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=128, num_heads=2, backend="hip", group_norm_weight=False, recurrent_weight_init="standard"))
    layer = layer.to(DEV).to(dtype).eval()
    assert layer.group_norm.weight is None and "group_norm.weight" not in layer.state_dict()
    layer.slstm_cell.keep_state_fp32 = True
    x = torch.randn(3, 6, 128, device=DEV).to(dtype)
    with torch.no_grad():
        want, states = layer(x, return_last_state=True)
        got = _lib.host().layer_forward(layer, layer.slstm_cell._native(), x, None, None, False, None)
        assert got is not None and torch.equal(got, want)
        if dtype == torch.bfloat16:  # (a float32 layer's step is not one of the native path's)
            token = x[:, :1].contiguous()
            want, want_states = layer.step(token, (states["conv_state"],), states["slstm_state"])  # (plans steps of 3 rows)
            got = _lib.host().layer_step(layer, layer.slstm_cell._native(), token, states["conv_state"], states["slstm_state"], *5 * [None])
            assert got is not None and torch.equal(got[0], want) and torch.equal(got[1]["slstm_state"], want_states["slstm_state"])
