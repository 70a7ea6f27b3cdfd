"""The sequence kernel with two workgroups per compute unit (``slstm_seq_pair_kernel``: bfloat16 heads of more than 512 units, and smaller
ones whose batch fills the device, 32 steps and more) at the sizes where it can go wrong: 33 workgroups per head and a last one half filled, row tiles of 4, 8 and 16 rows and two of
16, batches that leave rows over, more heads and rows than one launch holds, numbers of steps around its round of four tiles.

The same call in pieces of fewer than 32 steps runs in other kernels, which form every sum in the same order: the same bits."""
import numpy as np
import pytest
import torch

from oracle import slstm_oracle as so
from tests._util import geometric_reset_mask, make_problem
from tests.test_hip_parity import TOL_BF16, _check, _run_hip

pytestmark = pytest.mark.gpu

# B, T, NH, dh, rows of a workgroup
CASES = [
    (1, 33, 1, 520, 4),       # 33 workgroups, the last with 8 units
    (5, 32, 4, 1024, 4),
    (13, 35, 4, 1024, 8),     # ... row tiles of 8, the second with 5 rows
    (27, 34, 4, 768, 16),     # row tiles of 16, the second with 11 rows
    (40, 64, 4, 1024, 32),    # two row tiles, the last with 8 rows
    (61, 67, 4, 1000, 32),    # ... a last workgroup with 8 units, a row tile with 13 rows
    (70, 65, 4, 528, 32),     # ... and a second launch of 6 rows
    (61, 33, 4, 512, 16),     # head dims that fit an XCD at one workgroup per compute unit: one row tile in place of two
    (115, 34, 4, 248, 16),    # ... a last workgroup with 8 units, two chunks of K per wave
    (150, 65, 3, 328, 32),    # ... one launch in place of two
    (9, 36, 9, 536, 4),       # eight heads and one: two launches, the second in row tiles of 4
]


@pytest.mark.parametrize("B,T,NH,dh,rows", CASES)
@pytest.mark.parametrize("masked", [False, True], ids=["plain", "mask+state"])
def test_same_bits_as_in_short_pieces(B, T, NH, dh, rows, masked):
    print("case two workgroups per compute unit", B, T, NH, dh, masked, flush=True)
    wx, r, b, s0 = make_problem(91, B, T, NH, dh, bf16=True, with_state=masked)
    reset = geometric_reset_mask(6, B, T, 11) if masked else None
    h, s, status = _run_hip(wx, r, b, s0, reset, bf16=True)
    assert status["rows_per_workgroup"] == rows, status
    h_ref, s_ref = so.slstm_forward(wx, r, b, s0, reset)
    _check(h, s, h_ref, s_ref, TOL_BF16, status)
    state, parts = s0, []
    for t in range(0, T, 23):
        hp, state, _ = _run_hip(wx[:, t:t + 23], r, b, state, None if reset is None else reset[:, t:t + 23], bf16=True)
        parts.append(hp)
    np.testing.assert_array_equal(h, np.concatenate(parts))
    np.testing.assert_array_equal(s, state)


@pytest.mark.parametrize("B,T,NH,dh", [(3, 33, 1, 520), (11, 32, 4, 1024), (41, 34, 3, 768), (70, 33, 4, 528), (70, 32, 4, 504), (130, 33, 12, 144)])
def test_training_forward_leaves_the_same_coefficients(B, T, NH, dh):
    from xlstm_amd import functional as F

    print("case coefficients, two workgroups per compute unit", B, T, NH, dh, flush=True)
    dev = torch.device("cuda:0")
    torch.manual_seed(17)
    wx = torch.randn(B, T, 4 * NH * dh, device=dev).bfloat16()
    r = (torch.randn(NH, 4 * dh, dh, device=dev) / dh ** 0.5).bfloat16()
    bias = torch.randn(NH, 4, dh, device=dev)
    mask = torch.rand(B, T, device=dev) < 0.1

    def run(lo, hi, s0):
        x = wx[:, lo:hi].contiguous()
        coef = F.training_coefficients(x, NH)
        coef.zero_()
        h, s = F.slstm_forward(x, r, bias, s0, mask[:, lo:hi].contiguous(), train_coef=coef)
        return h, s, coef

    h, s, coef = run(0, T, None)
    h1, s1, c1 = run(0, T // 2, None)
    h2, s2, c2 = run(T // 2, T, s1)
    assert torch.equal(h, torch.cat([h1, h2])) and torch.equal(s, s2)
    # [T][row tiles of 4][heads][16 units][coefficients 0-3, 4-7, 8][row, unit]: rows and units that do not exist are nobody's
    sets = (B + 3) // 4 * NH * ((dh + 15) // 16)

    def elements(c, steps):
        c = c[:steps * sets * 576].view(steps, (B + 3) // 4, NH, (dh + 15) // 16, 576)
        v = torch.cat([c[..., :256].reshape(*c.shape[:4], 4, 16, 4), c[..., 256:512].reshape(*c.shape[:4], 4, 16, 4),
                       c[..., 512:].reshape(*c.shape[:4], 4, 16, 1)], dim=-1)
        v = v.permute(0, 1, 4, 2, 3, 5, 6).reshape(steps, (B + 3) // 4 * 4, NH, (dh + 15) // 16 * 16, 9)
        return v[:, :B, :, :dh]

    assert torch.equal(elements(coef, T), torch.cat([elements(c1, T // 2), elements(c2, T - T // 2)]))


def test_a_wait_that_runs_out_leaves_nan():
    """(as for the other sequence kernels: the caller's limit of one look per wait)"""
    B, T, NH, dh = 64, 64, 4, 1024
    print("case a wait that runs out, two workgroups per compute unit", flush=True)
    wx, r, b, _ = make_problem(18, B, T, NH, dh, bf16=True)
    for _ in range(20):
        h, s, status = _run_hip(wx, r, b, bf16=True, spin_limit=1)
        if status["aborted"]:
            break
    assert status["rows_per_workgroup"] == 32 and status["aborted"] == 1, status
    assert np.isnan(h).any() and np.isnan(s).any()
