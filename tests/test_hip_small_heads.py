"""Heads that stay in one compute unit (head dims up to 128): the forward and the reverse kernel at the edges of their
waves (16 units), row tiles (4 rows) and prefetch rings, against the oracles and bit for bit against the step kernel."""
import numpy as np
import pytest
import torch

from oracle import slstm_oracle as so
from tests._util import geometric_reset_mask, make_problem, max_err, r_ext_to_kernel

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rel(a, g):
    return float(np.abs(a - g).max() / max(1.0, np.abs(g).max()))


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("B,T,NH,dh,masked,opts", [
    (1, 1, 1, 8, False, {}), (4, 8, 2, 16, True, {}), (5, 9, 3, 24, True, {}), (3, 6, 1, 40, False, {}), (9, 7, 2, 64, True, {}),
    (2, 17, 5, 72, True, {}), (6, 13, 2, 96, False, {}), (7, 5, 1, 120, True, {}), (4, 25, 2, 128, True, {}),
    (5, 11, 2, 48, True, dict(recurrent_cut=True)), (5, 11, 2, 112, True, dict(recurrent_clipval=0.05)),
])
def test_small_heads_against_the_oracles(bf16, B, T, NH, dh, masked, opts):
    from xlstm_amd import functional as F

    print("case small heads", bf16, B, T, NH, dh, masked, opts, flush=True)
    H = NH * dh
    wx, r, b, s0 = make_problem(500 + dh, B, T, NH, dh, rscale=2.0, bf16=bf16, with_state=masked)
    reset = geometric_reset_mask(dh, B, T, max(2, T // 3)) if masked else None
    if reset is not None:
        reset[0, 0] = 0
    rng = np.random.default_rng(dh)
    d_h = rng.standard_normal((T, B, H)).astype(np.float32)
    d_sf = rng.standard_normal((4, B, H)).astype(np.float32)
    d_sf[3] = 0.0
    if bf16:
        d_h = torch.from_numpy(d_h).bfloat16().float().numpy()
        r = torch.from_numpy(r).bfloat16().float().numpy()
    dt = torch.bfloat16 if bf16 else torch.float32
    wx_t = torch.from_numpy(wx).to(DEV).to(dt)
    r_t, b_t = r_ext_to_kernel(torch.from_numpy(r)).to(DEV), torch.from_numpy(b).to(DEV)
    s0_t = torch.from_numpy(s0).to(DEV) if masked else None
    m_t = torch.from_numpy(reset).to(DEV) if masked else None
    coef = F.training_coefficients(wx_t, NH)
    h, s = F.slstm_forward(wx_t, r_t, b_t, s0_t, m_t, train_coef=coef)
    h_plain, s_plain = F.slstm_forward(wx_t, r_t, b_t, s0_t, m_t)
    st = s0_t
    for t in range(T):  # step by step: the same bits
        ht, st = F.slstm_forward(wx_t[:, t:t + 1], r_t.to(dt), b_t, st, m_t[:, t:t + 1] if masked else None, step=True)
        assert torch.equal(ht[0], h[t]) and torch.equal(ht[0], h_plain[t]), t
    assert torch.equal(st, s) and torch.equal(st, s_plain)
    h_ref, s_ref = so.slstm_forward(wx, r, b, s0, reset)
    tol = 2e-2 if bf16 else 1e-5
    assert max_err(h.float().cpu().numpy(), h_ref) <= tol and max_err(s.cpu().numpy(), s_ref) <= tol
    # the gradient of h as a layer's norm hands it back ([B, S, H] in memory), with and without the forward's coefficients
    d_h_t = torch.from_numpy(d_h).to(DEV).to(dt).transpose(0, 1).contiguous().transpose(0, 1)
    o = so.slstm_backward(wx, r, b, s0, reset, d_h, d_sf, **opts)
    o = (o[0], r_ext_to_kernel(torch.from_numpy(o[1])).numpy(), o[2], o[3])
    for c in (coef, None):
        got = F.slstm_backward(wx_t, r_t, b_t, s0_t, m_t, h, d_h_t, torch.from_numpy(d_sf).to(DEV), coef=c, **opts)
        errs = [_rel(x.cpu().numpy(), y) for x, y in zip(got, o)]
        print(errs, flush=True)
        assert all(np.isfinite(e) and e <= tol for e in errs), errs
    if bf16:
        short = F.slstm_backward(wx_t, r_t, b_t, s0_t, m_t, h, d_h_t, torch.from_numpy(d_sf).to(DEV), coef=coef, d_wx_dtype=dt, **opts)
        assert torch.equal(short[0], got[0].to(dt)) and torch.equal(short[3], got[3])


@pytest.mark.parametrize("bf16,B,NH,dh", [(True, 64, 40, 128), (True, 33, 33, 128), (True, 40, 72, 64), (False, 40, 72, 64), (True, 65, 129, 24)])
def test_more_heads_than_one_launch_holds(bf16, B, NH, dh):
    """The heads in front run in the kernel of four row tiles, the last few in one compute unit each: every head against the
    oracle and bit for bit against the step kernel."""
    from xlstm_amd import functional as F

    print("case heads in several launches", bf16, B, NH, dh, flush=True)
    T = 4
    wx, r, b, s0 = make_problem(700 + dh, B, T, NH, dh, rscale=2.0, bf16=bf16, with_state=True)
    reset = geometric_reset_mask(dh, B, T, 3)
    if bf16:
        r = torch.from_numpy(r).bfloat16().float().numpy()
    dt = torch.bfloat16 if bf16 else torch.float32
    wx_t = torch.from_numpy(wx).to(DEV).to(dt)
    r_t, b_t = r_ext_to_kernel(torch.from_numpy(r)).to(DEV), torch.from_numpy(b).to(DEV)
    s0_t, m_t = torch.from_numpy(s0).to(DEV), torch.from_numpy(reset).to(DEV)
    ws = F.workspace_for(B, T, NH, dh, DEV)
    h, s = F.slstm_forward(wx_t, r_t, b_t, s0_t, m_t, workspace=ws)
    status = F.read_status(ws)
    assert status["launches"] > 1 and status["rows_per_workgroup"] == 4 and status["aborted"] == 0, status
    st = s0_t
    for t in range(T):
        ht, st = F.slstm_forward(wx_t[:, t:t + 1], r_t.to(dt), b_t, st, m_t[:, t:t + 1], step=True)
        assert torch.equal(ht[0], h[t]), t
    assert torch.equal(st, s)
    h_ref, s_ref = so.slstm_forward(wx, r, b, s0, reset)
    tol = 2e-2 if bf16 else 1e-5
    assert max_err(h.float().cpu().numpy(), h_ref) <= tol and max_err(s.cpu().numpy(), s_ref) <= tol
