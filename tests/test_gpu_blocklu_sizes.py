"""Batched LU at every kind of block size: sizes compiled with m constant and
sizes between them (m at run time in the next row length), around the lane
groups' edges.  FP64 factors, pivots and solutions are the oracle's
(oracle_block_getrf / _getrs) bit for bit; FP32 factors and pivots are those of
the same algorithm in numpy float32, the solve from them in float64.  The
blocks hold what the kernels treat apart: dense rows, rows full of zeros of
both signs, tied pivots, a NaN, an infinity, and entries far outside the range
of the reciprocal-based quotients."""
import ctypes as C

import numpy as np
import pytest

from sundials_amd import _lib
from helpers import dp, gpu_get, gpu_vec
from test_gpu_blocklu import _gpu_matrix, _gpu_matrix_values, _setup_run, _to_blockmajor

pytestmark = pytest.mark.gpu

# both sides of every row length, and sizes with a kernel of their own
SIZES = [2, 5, 9, 10, 11, 12, 13, 15, 16, 17, 20, 21, 23, 24, 25, 28, 29, 31, 32, 33, 40, 41, 47, 48,
         49, 56, 57, 63, 64]


def _cases(m, seed):
    rng = np.random.default_rng(seed)
    A = rng.uniform(-1, 1, (9, m, m))
    A[1] *= rng.random((m, m)) < 0.3              # sparse, filling in
    A[1] += np.diag(rng.uniform(1, 2, m))
    A[2] = np.where(rng.random((m, m)) < 0.3, A[2], -0.0) + np.diag(rng.uniform(1, 2, m))
    A[3] = np.sign(A[3]) + 2.0 * m * np.eye(m)[:, rng.permutation(m)]  # tied entries
    A[4, :, 0] = 0.5                              # a tied column
    A[5, m // 2, 0] = np.nan
    A[6, m - 1, m - 1] = np.inf
    A[7] = (np.eye(m) * 2.0 ** -900 if m % 2 else np.eye(m) * 2.0 ** 900)  # quotients by division
    b = rng.uniform(-1, 1, (9, m))
    b[8] *= rng.random(m) < 0.5
    b[8, 0] = -0.0
    return A, b


def _numpy_getrf(A, T):
    """SUNDlsMat_denseGETRF (sundials_dense.c:85-143) in precision T."""
    a = A.astype(T)
    m = len(a)
    p = np.zeros(m, np.int64)
    with np.errstate(all="ignore"):
        for k in range(m):
            l = k
            for i in range(k + 1, m):
                if abs(a[i, k]) > abs(a[l, k]):
                    l = i
            p[k] = l
            if l != k:
                a[[k, l]] = a[[l, k]]
            a[k + 1:, k] *= T(1) / a[k, k]
            for j in range(k + 1, m):
                if a[k, j] != 0:
                    a[k + 1:, j] -= a[k, j] * a[k + 1:, k]
    return a, p


def _solve(core, hip, ctx, A, b, prec):
    nb, m, _ = A.shape
    y = gpu_vec(ctx, np.zeros(nb * m))
    M = _gpu_matrix(hip, ctx, y, A)
    LS = hip.SUNLinSol_Mi355BlockLU(y, M, prec, ctx)
    assert LS and core.SUNLinSolInitialize(LS) == 0
    assert core.SUNLinSolSetup(LS, M) == 0
    F = _gpu_matrix_values(hip, M, nb, m)
    piv = np.zeros(nb * m, np.int32)
    assert hip.SUNLinSol_Mi355BlockLU_GetPivots(LS, piv.ctypes.data_as(C.POINTER(C.c_int))) == 0
    gb, gx = gpu_vec(ctx, b.ravel()), gpu_vec(ctx, np.zeros(nb * m))
    assert core.SUNLinSolSolve(LS, M, gx, gb, 0.0) == 0
    x = gpu_get(gx)
    core.SUNLinSolFree(LS)
    core.SUNMatDestroy(M)
    for v in (y, gb, gx):
        core.N_VDestroy(v)
    return F, piv.reshape(nb, m), x.reshape(nb, m)


@pytest.fixture
def ctx():
    c = _lib.new_context()
    yield c
    _lib.free_context(c)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("m", SIZES)
def test_every_size_follows_the_dense_solver(ctx, m, prec):
    core, hip, orc = _lib.core(), _lib.hip(), _lib.load_oracle()
    A, b = _cases(m, 100 * m + prec)
    if prec:
        A = np.delete(A, 7, axis=0)  # 2^+-900 has no single-precision value
        b = np.delete(b, 7, axis=0)
    nb = len(A)
    F, piv, x = _solve(core, hip, ctx, A, b, prec)
    for k in range(nb):
        a, p = _numpy_getrf(A[k], np.float32 if prec else np.float64)
        finite = np.isfinite(A[k]).all()
        assert np.array_equal(piv[k], p), ("pivots", k)
        if prec == 0:
            o = _to_blockmajor(A[k:k + 1]).copy()
            q = np.zeros(m, np.int64)
            assert orc.oracle_block_getrf(dp(o), m, q.ctypes.data_as(C.POINTER(C.c_int64))) == 0
            assert np.array_equal(F[k * m * m:(k + 1) * m * m], o, equal_nan=True), ("factor", k)
            assert np.array_equal(p, q)
        # the solve in float64 from these factors, by the oracle
        o = np.ascontiguousarray(a.T.astype(np.float64)).ravel()
        r = b[k].copy()
        orc.oracle_block_getrs(dp(o), m, p.ctypes.data_as(C.POINTER(C.c_int64)), dp(r))
        assert np.array_equal(x[k], r, equal_nan=not finite), ("solve", k)


def test_scale_add_i_over_several_pairs_per_thread(ctx):
    """Beyond 2^25 elements a thread takes a pair, then the one a whole grid
    further, at another place of its block (2^25 mod 441 = 65); the total is
    odd, so the last element stands alone."""
    core, hip = _lib.core(), _lib.hip()
    nb, m, c = 80001, 21, -0.3125
    y = gpu_vec(ctx, np.zeros(1))
    M = hip.SUNMatrix_Mi355BlockDense(nb, m, hip.N_VGetStream_Mi355(y), ctx)
    a = np.random.default_rng(21).uniform(-1, 1, nb * m * m)
    C.memmove(hip.SUNMatrix_Mi355BlockDense_HostData(M), dp(a), 8 * a.size)
    assert hip.SUNMatrix_Mi355BlockDense_CopyToDevice(M) == 0
    assert core.SUNMatScaleAddI(c, M) == 0
    a *= c
    a.reshape(nb, m * m)[:, ::m + 1] += 1.0
    assert np.array_equal(_gpu_matrix_values(hip, M, nb, m), a)
    core.SUNMatDestroy(M)
    core.N_VDestroy(y)


ONE_PASS = {*range(1, 11), 12, 16, 24, 32, 48, 64}  # sizes compiled with m constant


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("m", range(1, 65))
def test_one_pass_calls_at_every_size(ctx, m, prec):
    """The one-pass setup and solve either do the separate calls' work bit for
    bit or decline with everything as it was: a setup that reports success has
    factored."""
    core, hip = _lib.core(), _lib.hip()
    nb = 5
    J = np.random.default_rng(m).uniform(-1, 1, (nb, m, m)) * 4.0 / m
    ref = _setup_run(core, hip, ctx, J, prec, 0, False, -0.25)
    y = gpu_vec(ctx, np.zeros(nb * m))
    MA, MJ = _gpu_matrix(hip, ctx, y, np.zeros_like(J)), _gpu_matrix(hip, ctx, y, J)
    LS = hip.SUNLinSol_Mi355BlockLU(y, MA, prec, ctx)
    assert core.SUNLinSolInitialize(LS) == 0
    flag = hip.SUNLinSol_Mi355BlockLUSetupScaled(LS, MA, MJ, -0.25, 0)
    b = np.random.default_rng(5).uniform(-1, 1, nb * m)  # the right-hand side of _setup_run
    gb = gpu_vec(ctx, b)
    if m in ONE_PASS:
        assert flag == 0
        assert np.array_equal(_gpu_matrix_values(hip, MA, nb, m), ref[1])
        assert hip.SUNLinSol_Mi355BlockLUSolveScaled(LS, MA, gb, 1.0) == 0
        assert np.array_equal(gpu_get(gb), ref[3])
    else:
        incompatible = -9998
        assert flag == incompatible
        assert not _gpu_matrix_values(hip, MA, nb, m).any()
        assert hip.SUNLinSol_Mi355BlockLUSolveScaled(LS, MA, gb, 1.0) == incompatible
        assert np.array_equal(gpu_get(gb), b)
    core.SUNLinSolFree(LS)
    for M in (MA, MJ):
        core.SUNMatDestroy(M)
    for v in (y, gb):
        core.N_VDestroy(v)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("m", [11, 21, 33, 41, 49, 57, 63, 64])
def test_zero_pivot_in_every_group_width(ctx, m, prec):
    """A zero column, which stays one through the elimination, in groups of 16, 32 and
    64 lanes with m at run time and in 64 with m constant: the first failing
    block's column is reported, and the other blocks' factors and pivots are
    those of the dense solver."""
    core, hip, orc = _lib.core(), _lib.hip(), _lib.load_oracle()
    nb, bad, col = 6, 3, m - 2
    A = np.random.default_rng(m).uniform(-1, 1, (nb, m, m))
    A[bad, :, col] = 0.0
    A[bad + 1, :, m - 1] = -0.0
    y = gpu_vec(ctx, np.zeros(nb * m))
    M = _gpu_matrix(hip, ctx, y, A)
    LS = hip.SUNLinSol_Mi355BlockLU(y, M, prec, ctx)
    assert core.SUNLinSolSetup(LS, M) == 808  # SUNLS_LUFACT_FAIL
    assert core.SUNLinSolLastFlag(LS) == bad * m + col + 1
    piv = np.zeros(nb * m, np.int32)
    assert hip.SUNLinSol_Mi355BlockLU_GetPivots(LS, piv.ctypes.data_as(C.POINTER(C.c_int))) == 0
    F = _gpu_matrix_values(hip, M, nb, m).reshape(nb, m * m)
    for k in range(nb):
        a, p = _numpy_getrf(A[k], np.float32 if prec else np.float64)
        upto = {bad: col, bad + 1: m - 1}.get(k, m)  # columns before the zero pivot
        assert np.array_equal(piv.reshape(nb, m)[k][:upto], p[:upto]), k
        if prec == 0:
            o = _to_blockmajor(A[k:k + 1]).copy()
            q = np.zeros(m, np.int64)
            rc = orc.oracle_block_getrf(dp(o), m, q.ctypes.data_as(C.POINTER(C.c_int64)))
            assert rc == {bad: col + 1, bad + 1: m}.get(k, 0)
            if rc == 0:
                assert np.array_equal(F[k], o), k
    core.SUNLinSolFree(LS)
    core.SUNMatDestroy(M)
    core.N_VDestroy(y)
