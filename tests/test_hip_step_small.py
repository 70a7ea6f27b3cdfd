"""The decode step of small batches (16 rows x 16 units per workgroup) against the float64 oracle and, bit for bit, against the
same token inside a sequence call: head dims around the unit tiles and the ends of the K ranges, rows around the row tiles,
with and without a state, a mask, the bfloat16 operand of the step before."""
import numpy as np
import pytest
import torch

from oracle import slstm_oracle as so
from tests._util import make_problem, max_err, r_ext_to_kernel

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("bf16,B,NH,dh", [
    (True, 1, 1, 8), (True, 17, 3, 24), (True, 16, 2, 128), (True, 5, 2, 136), (True, 33, 1, 248), (True, 3, 4, 256), (True, 2, 1, 264),
    (True, 15, 2, 512), (True, 4, 1, 520), (True, 1, 2, 1024), (False, 1, 2, 8), (False, 18, 1, 56), (False, 7, 2, 64), (False, 16, 1, 72),
    (False, 2, 3, 128), (False, 31, 1, 200), (False, 1, 2, 256), (False, 3, 1, 264), (False, 2, 2, 512),
])
def test_step_of_a_small_batch(bf16, B, NH, dh):
    from xlstm_amd import functional as F

    print("case small step", bf16, B, NH, dh, flush=True)
    T = 3
    wx, r, b, _ = make_problem(dh + B, B, T, NH, dh, bf16=bf16)
    dt = torch.bfloat16 if bf16 else torch.float32
    x = torch.from_numpy(wx).to(DEV, dt)
    r_t = r_ext_to_kernel(torch.from_numpy(r)).to(DEV).to(dt)
    b_t = torch.from_numpy(b).to(DEV)
    rng = np.random.default_rng(dh)
    reset = rng.random((B, T)) < 0.4
    for mask in (None, reset):
        m = None if mask is None else torch.from_numpy(mask).to(DEV)
        _run(F, so, x, wx, r_t, r, b_t, b, mask, m, T, bf16)


def _run(F, so, x, wx, r_t, r, b_t, b, mask, m, T, bf16):
    h_seq, s_seq = F.slstm_forward(x, r_t, b_t, None, m)
    h_ref, s_ref = so.slstm_forward(wx, r, b, None, mask)
    tol = 2e-2 if bf16 else 1e-5  # (the bars of the cell's parity tests; float32: K products of order 1 / sqrt(K) and three steps of gating, a few 2^-24 each)
    state, h_prev = None, None
    for t in range(T):
        mt = None if m is None else m[:, t:t + 1]
        plain = F.slstm_forward(x[:, t:t + 1], r_t, b_t, state, mt, step=True)
        if h_prev is not None and bf16:
            hinted = F.slstm_forward(x[:, t:t + 1], r_t, b_t, state, mt, step=True, h_prev=h_prev)
            assert torch.equal(plain[0], hinted[0]) and torch.equal(plain[1], hinted[1])
        h, state = plain
        h_prev = h
        assert torch.equal(h[0], h_seq[t]), t
    assert torch.equal(state, s_seq)
    assert max_err(h_seq.float().cpu().numpy(), h_ref) <= tol and max_err(state.cpu().numpy(), s_ref) <= tol
