"""A layer's decoded token in one kernel up to its hidden state against the kernels of its parts called in a row: the same bits,
at the edges of its row tiles, unit tiles and of the splits it is launched in."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B,NH,dh,extra", [
    (1, 1, 64, {}),                                  # half of the four waves have no share of K
    (17, 4, 64, dict(state=False)),                  # a row behind a tile; no inputs before the first
    (16, 3, 128, dict(bias=False)), (33, 2, 192, {}),  # K ends inside the third and fourth share
    (260, 1, 256, {}), (40, 8, 256, {}),             # one compute unit each, and 32 units a workgroup
    (100, 8, 256, dict(state=False)),                # several row tiles a workgroup, the last ragged
    (600, 2, 128, {}), (70, 16, 192, {}),            # the same with one k-step, and with K inside a share
    (1040, 1, 64, {}),                               # more row tiles than rows of the grid, waves without a share
    (5, 2, 320, {}), (33, 4, 512, dict(hint=True)),  # four k-steps a share, 16 and 32 units
    (3, 1, 1024, {}), (7, 2, 128, dict(K=3)),        # the kernels of the parts
])
@pytest.mark.parametrize("hint", [False, True])
def test_layer_step_equals_its_parts(B, NH, dh, extra, hint):
    from xlstm_amd import functional as hipF
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case layer step", B, NH, dh, extra, hint, flush=True)
    D, K = NH * dh, extra.get("K", 4)
    torch.manual_seed(B + dh)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=D, num_heads=NH, conv1d_kernel_size=K, backend="hip", recurrent_weight_init="standard"))
    layer = layer.to(DEV).bfloat16().eval()
    if extra.get("bias") is False:
        layer.conv1d.conv.bias = None
    layer.slstm_cell.keep_state_fp32 = True
    conv = layer.conv1d.conv
    before = torch.randn(B, K - 1, D, device=DEV).bfloat16() if extra.get("state", True) else None
    s = torch.randn(4, B, D, device=DEV)
    s[0].tanh_()
    s[2] = s[2].abs() + 1.0
    h_prev = s[0:1].bfloat16() if hint else None
    x = torch.randn(3, B, 1, D, device=DEV).bfloat16()
    with torch.no_grad():
        layer.slstm_cell.step(torch.zeros(B, 1, 4 * D, device=DEV, dtype=torch.bfloat16), s)  # (plans steps of B rows)
        state, hp, ring = s, h_prev, before
        got_state, got_ring = s, (before,) if before is not None else None
        for t in range(3):
            out, st = layer.step(x[t], conv_state=got_ring, slstm_state=got_state, h_prev=h_prev if t == 0 else None)
            new_ring = torch.full((B, K, D), 7.0, device=DEV, dtype=torch.bfloat16)
            x_conv = hipF.causal_conv_silu(x[t], conv.weight, conv.bias, ring, ring_out=new_ring)
            wx = hipF.headwise_gates(x[t], x_conv, (layer.fgate.weight, layer.igate.weight, layer.zgate.weight, layer.ogate.weight), NH)
            h, new_state = hipF.slstm_forward(wx, layer.slstm_cell._recurrent_kernel_, layer.slstm_cell._bias_.float().view(NH, 4, dh), state,
                                              step=True, h_prev=hp)
            want = hipF.headwise_group_norm(h.view(1, B, NH, dh).permute(1, 2, 0, 3), layer.group_norm.weight, layer.group_norm.eps)
            assert torch.equal(st["slstm_state"], new_state), t
            assert torch.equal(st["conv_state"][0], new_ring), t
            assert torch.equal(out, want), t
            got_state, got_ring = st["slstm_state"], st["conv_state"]
            state, hp, ring = new_state, None, new_ring[:, 1:]
    assert layer.slstm_cell.last_status()["step_kernel"] == 1


def test_layer_step_refuses_what_its_parts_refuse():
    import ctypes

    from xlstm_amd import _lib

    print("case layer step refusals", flush=True)
    lib = _lib.load()
    assert lib.xs_layer_step(None) == -1
    a = _lib.LayerStepArgs()
    a.cell.B, a.cell.T, a.cell.NH, a.cell.dh, a.K = 2, 1, 2, 64, 4
    assert lib.xs_layer_step(ctypes.byref(a)) == -3  # float32
    a.cell.wx_dtype = a.cell.r_dtype = _lib.XS_BF16
    a.cell.dh = 96
    assert lib.xs_layer_step(ctypes.byref(a)) == -5
    a.cell.dh = 64
    assert lib.xs_layer_step(ctypes.byref(a)) == -5  # no state
    a.cell.s0 = 0x100000
    assert lib.xs_layer_step(ctypes.byref(a)) == -1  # x, ring_out
    ring = torch.zeros(2, 4, 128, dtype=torch.bfloat16, device=DEV)
    s0, s1 = torch.zeros(4, 2, 128, device=DEV), torch.zeros(4, 2, 128, device=DEV)
    r, b, ws = torch.zeros(2, 256, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(2, 4, 64, device=DEV), torch.zeros(1 << 22, dtype=torch.uint8, device=DEV)
    w = torch.zeros(2, 64, 64, dtype=torch.bfloat16, device=DEV)
    row = torch.zeros(2, 2, 128, dtype=torch.bfloat16, device=DEV)
    c = a.cell
    c.s0, c.s_out, c.r, c.bias, c.h_out, c.workspace = (t.data_ptr() for t in (s0, s1, r, b, row[0], ws))
    c.workspace_bytes = ws.numel()
    a.x, a.ring_out, a.conv_state, a.conv_w = row[1].data_ptr(), ring.data_ptr(), ring.data_ptr(), w.data_ptr()
    for i in range(4):
        a.gate_w[i] = w.data_ptr()
    a.conv_state_stride_b = 4 * 128
    assert lib.xs_layer_step(ctypes.byref(a)) == -2 and b"overlap" in lib.xs_last_error()  # the ring in place
    a.conv_state, a.x = None, ring.data_ptr()
    assert lib.xs_layer_step(ctypes.byref(a)) == -2 and b"overlap" in lib.xs_last_error()
    a.x, a.conv_w = row[1].data_ptr(), w.data_ptr() + 2
    assert lib.xs_layer_step(ctypes.byref(a)) == -4
    a.conv_w, a.K = w.data_ptr(), 3
    assert lib.xs_layer_step(ctypes.byref(a)) == -5 and not lib.xs_layer_step_fits(2, 2, 64, 3)  # three taps: its parts
    a.K = 4
    # h_out or s_out in the memory of x or of the taps (rows of 2 x 128, taps of 3 x 128 each), at both ends
    free, taps = torch.zeros(8, 2, 128, dtype=torch.bfloat16, device=DEV), torch.zeros(2, 3, 128, dtype=torch.bfloat16, device=DEV)
    h, s_out, x = c.h_out, c.s_out, a.x
    for moved in (dict(h=x), dict(h=x + 496), dict(x=s_out), dict(x=s_out + 16 * 256 - 16), dict(taps=h + 496), dict(taps=h - 3 * 512 + 16),
                  dict(taps=s_out + 16 * 256 - 16)):
        c.h_out, a.x, a.conv_state = moved.get("h", h), moved.get("x", x), moved.get("taps")
        a.conv_state_stride_b = 0
        assert lib.xs_layer_step(ctypes.byref(a)) == -2 and b"overlap" in lib.xs_last_error(), moved
    c.h_out, a.x, a.conv_state = free[0].data_ptr(), free[1].data_ptr(), taps.data_ptr()  # next to each other
    for at, error in ((a.x + 496, -2), (taps.data_ptr() + 3 * 512 - 16, -2), (free[2].data_ptr() + 8, -4)):
        a.x_out = at
        assert lib.xs_layer_step(ctypes.byref(a)) == error
    a.x_out = free[2].data_ptr()
    free[1].fill_(3.0)
    assert lib.xs_layer_step(ctypes.byref(a)) == 0 and lib.xs_layer_step_fits(2, 2, 64, 4)
    torch.cuda.synchronize()
    assert torch.equal(free[2], free[1]) and not free[3].any()


@pytest.mark.parametrize("shared", ["h over x", "state over x", "h over taps", "state over taps"])
def test_buffers_that_share_memory_give_what_the_parts_give(shared):
    """h_out or slstm_state_out in the memory of x or of the convolution's state: the convolution and the projections have read both before
    the cell's step writes."""
    from xlstm_amd.layer import sLSTMLayer, sLSTMLayerConfig

    print("case layer step shared", shared, flush=True)
    B, NH, dh = 48, 4, 256
    D = NH * dh
    torch.manual_seed(1)
    layer = sLSTMLayer(sLSTMLayerConfig(embedding_dim=D, num_heads=NH, backend="hip", recurrent_weight_init="standard")).to(DEV).bfloat16().eval()
    layer.slstm_cell.keep_state_fp32 = True
    x, taps = torch.randn(B, 1, D, device=DEV).bfloat16(), torch.randn(B, 3, D, device=DEV).bfloat16()
    state = torch.rand(4, B, D, device=DEV) + 0.5
    memory = torch.zeros(16 * B * D, dtype=torch.uint8, device=DEV)  # (as large as a state)

    def at(t):  # t's values at the start of that memory
        v = memory[:t.numel() * t.element_size()].view(t.dtype).view(t.shape)
        v.copy_(t)
        return v

    with torch.no_grad():
        layer.slstm_cell.step(torch.zeros(B, 1, 4 * D, device=DEV, dtype=torch.bfloat16), state)  # (plans steps of B rows)
        want, want_st = layer.step(x, conv_state=(taps,), slstm_state=state)
        tokens, ring = (at(x), taps) if "x" in shared else (x, at(taps))
        out = {"h_out": memory[:2 * B * D].view(torch.bfloat16).view(1, B, D)} if shared.startswith("h") else \
              {"slstm_state_out": memory.view(torch.float32).view(4, B, D)}
        got, got_st = layer.step(tokens, conv_state=(ring,), slstm_state=state, **out)
    assert torch.equal(got, want) and torch.equal(got_st["slstm_state"], want_st["slstm_state"])
    assert torch.equal(got_st["conv_state"][0], want_st["conv_state"][0])
