"""Batched integrator where the solves' quotients leave the range in which the
diagonal's reciprocal gives the correctly rounded quotient, so that the sweep
with divisions runs: in every other system some species start at zero and all
their reactions are 1e-140 times slower, which keeps their Newton residuals
non-zero and below 2^-400.  FP64: the oracle's run bit for bit.  FP32 factors
(groups of up to 16 lanes, whose solves share that code): the other species and
every counter are those of the run in which the slow reactions do not run at
all, where the quotients need no division -- what the slow species add to the
other species' sums and norms is below half an ulp of them."""
import numpy as np
import pytest

from batch_util import free_batch, make_batch, run_device, run_oracle, system_slices

pytestmark = pytest.mark.gpu

LU_FP64, LU_FP32 = 0, 1
NSYS = 40


def _slow_species(b, factor):
    """Scale the rates of every reaction of the last species of every other
    cell by `factor` and start these species at zero.  Returns the bucket's
    species outside those reactions' reach (touched by other reactions too)."""
    p = b.contents.bucket[0].contents
    m, R, n = p.m, p.R, p.ncells
    idx = np.ctypeslib.as_array(p.idx, shape=(R, 4))
    slow = np.arange(m) >= m - max(1, m // 8)
    hit = slow[idx].any(axis=1)
    for a in (p.kf, p.kb):
        np.ctypeslib.as_array(a, shape=(n, R))[::2, hit] *= factor
    np.ctypeslib.as_array(p.y0, shape=(n, m))[::2, slow] = 0.0
    others = np.zeros(m, bool)
    others[idx[~hit].ravel()] = True
    return slow, others & ~slow


def _by_cell(b, y):
    m = b.contents.bucket[0].contents.m
    out = np.zeros((NSYS, m))
    for s, (_, c, _, off) in enumerate(system_slices(b)):
        out[c] = y[off:off + m]
    return out


@pytest.mark.parametrize("m", [3, 4, 5, 8, 12, 16, 24, 32, 48, 64])
def test_fp64_division_sweep_bitwise_vs_oracle(m):
    b = make_batch(NSYS, 9300 + m, m_values=(m,), weights=(1.0,))
    try:
        slow, _ = _slow_species(b, 1e-140)
        y_ref, c_ref, rc, _ = run_oracle(b)
        assert rc == 0
        tail = np.abs(_by_cell(b, y_ref)[::2, slow])
        assert tail.max() < 2.0 ** -400 and (tail > 0).any(axis=1).all()
        y, cnt, rc, _ = run_device(b, LU_FP64)
        assert rc == 0
        assert np.array_equal(cnt, c_ref)
        assert np.array_equal(y, y_ref)
    finally:
        free_batch(b)


@pytest.mark.parametrize("m", [4, 8, 12, 16])
def test_fp32_division_sweep_changes_no_other_species(m):
    runs = []
    for factor in (1e-140, 0.0):
        b = make_batch(NSYS, 9300 + m, m_values=(m,), weights=(1.0,))
        try:
            slow, others = _slow_species(b, factor)
            y, cnt, rc, _ = run_device(b, LU_FP32)
            assert rc == 0
            runs.append((_by_cell(b, y), cnt))
        finally:
            free_batch(b)
    (y, cnt), (y0, cnt0) = runs
    assert others.any() and (np.abs(y[::2, slow]) > 0).any(axis=1).all()
    assert not y0[::2, slow].any()
    assert np.array_equal(cnt, cnt0)
    assert np.array_equal(y[:, others], y0[:, others])
