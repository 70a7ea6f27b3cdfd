"""The parameter gradients from gate deltas in bf16 (``xs_slstm_backward_params`` with ``d_wx_dtype`` XS_BF16) against float64
sums of the same operands: head dims around the tiles of 64, 128 and 256 columns, sequences around the chunks of 32 steps,
slices of one and of several chunks, document starts, an initial state, strides.

The products of bf16 values are exact in float32; n of them added in any order are off by at most n 2^-24 of the sum of their
magnitudes (twice that is allowed)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B,T,NH,dh,state,mask,gap", [
    (1, 1, 1, 8, False, False, 0), (1, 2, 3, 64, True, True, 0), (3, 31, 2, 72, True, False, 8), (2, 32, 1, 128, False, True, 0),
    (5, 33, 2, 136, True, True, 0), (35, 3, 1, 192, True, True, 0), (4, 65, 4, 256, True, True, 16), (2, 200, 1, 264, False, True, 0),
    (3, 40, 2, 512, True, False, 0), (33, 70, 1, 1024, True, True, 0), (2, 5, 8, 640, False, False, 0),
])
def test_parameter_gradients_from_bf16_deltas(B, T, NH, dh, state, mask, gap):
    from xlstm_amd import _lib

    print("case parameter slabs", B, T, NH, dh, state, mask, gap, flush=True)
    g = torch.Generator(device="cpu").manual_seed(dh + T)
    H = NH * dh
    d = torch.randn(B, T, 4 * H + gap, generator=g).bfloat16()
    h = torch.randn(T, B, H, generator=g).bfloat16()
    s0 = torch.randn(4, B, H, generator=g)
    starts = torch.rand(B, T, generator=g) < 0.2
    dd, hd, sd, md = d.to(DEV), h.to(DEV), s0.to(DEV), starts.to(DEV).view(torch.uint8)
    d_r = torch.full((NH, 4 * dh, dh), 7.0, device=DEV)
    d_bias = torch.full((NH, 4, dh), 7.0, device=DEV)
    a = _lib.SlstmBwdArgs()
    a.B, a.T, a.NH, a.dh = B, T, NH, dh
    a.dtype = a.d_wx_dtype = _lib.XS_BF16
    a.d_wx, a.d_wx_stride_b, a.d_wx_stride_t = dd.data_ptr(), dd.stride(0), dd.stride(1)
    a.h_out = hd.data_ptr()
    a.s0 = sd.data_ptr() if state else None
    a.reset, a.reset_stride_b = (md.data_ptr(), T) if mask else (None, 0)
    a.d_r, a.d_bias = d_r.data_ptr(), d_bias.data_ptr()
    a.stream = torch.cuda.current_stream().cuda_stream
    assert _lib.load().xs_slstm_backward_params(ctypes.byref(a)) == 0, _lib.last_error()
    torch.cuda.synchronize()
    y = torch.zeros(T, B, H, dtype=torch.float64)
    y[1:] = h[:-1].double()
    if state:
        y[0] = s0[0].bfloat16().double()
    if mask:
        y[starts.t()] = 0.0
    dv = d[..., : 4 * H].double().reshape(B * T, 4, NH, dh).permute(2, 1, 3, 0).reshape(NH, 4 * dh, B * T)
    yv = y.transpose(0, 1).reshape(B * T, NH, dh).permute(1, 0, 2)
    n = B * T
    for got, want, size in ((d_r, dv @ yv, dv.abs() @ yv.abs()),
                            (d_bias.reshape(NH, 4 * dh), dv.sum(-1), dv.abs().sum(-1))):
        assert ((got.cpu().double() - want).abs() <= 2 * n * 2.0 ** -24 * size + 1e-30).all()
