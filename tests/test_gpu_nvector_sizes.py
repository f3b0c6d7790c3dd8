"""Vector ops at the lengths where their launches change: one to several
element pairs per lane (streaming ops), reductions folded on the host up to
256 workgroups and by the finish kernel beyond, Gram-Schmidt steps of one and
more passes of up to 12 vectors, and a reduction that outlasts the host's
watch on its result slot.  Elementwise results equal numpy's float64 bit for
bit; a sum of n terms in any order is within n * 2^-53 * sum |terms| of the
exact one (twice that here: the products round too)."""
import ctypes as C
import math

import numpy as np
import pytest

from sundials_amd import _lib
from helpers import dp, gpu_get, gpu_vec, vec_array

pytestmark = pytest.mark.gpu

# 256 and 257 workgroups of 4096 (one or two inputs) and of 2048 elements
# (three); the streaming thresholds 2 * 4 * 256 * 256 and that times 8 elements
EDGES = [1, 2, 4095, 4097, 524287, 524288, 524290, 526337, 1048576, 1048577, 1052673, 4194303, 4194306]


@pytest.fixture
def ctx():
    c = _lib.new_context()
    yield c
    _lib.free_context(c)


def _close(got, terms):
    exact = math.fsum(terms)
    return abs(got - exact) <= 2 * len(terms) * 2.0 ** -53 * math.fsum(np.abs(terms)) + 0.0


@pytest.mark.parametrize("n", EDGES)
def test_launch_edges(ctx, n):
    core = _lib.core()
    rng = np.random.default_rng(n)
    x, y, w = rng.standard_normal(n), rng.standard_normal(n), rng.uniform(0.5, 2, n)
    vx, vy, vw, vz = (gpu_vec(ctx, a) for a in (x, y, w, np.zeros(n)))
    idv = np.where(rng.random(n) < 0.7, 1.0, 0.0)
    vi = gpu_vec(ctx, idv)
    core.N_VLinearSum(0.3, vx, -0.7, vy, vz)
    assert np.array_equal(gpu_get(vz), 0.3 * x + (-0.7) * y)
    core.N_VScale(-2.5, vx, vz)
    assert np.array_equal(gpu_get(vz), -2.5 * x)
    core.N_VDiv(vx, vw, vz)
    assert np.array_equal(gpu_get(vz), x / w)
    c = (C.c_double * 3)(0.5, -1.25, 3.0)
    assert core.N_VLinearCombination(3, c, vec_array([vx, vy, vw]), vz) == 0
    assert np.array_equal(gpu_get(vz), (0.5 * x + -1.25 * y) + 3.0 * w)
    assert _close(core.N_VDotProd(vx, vy), x * y)
    assert _close(core.N_VL1Norm(vx), np.abs(x))
    assert core.N_VMaxNorm(vx) == np.abs(x).max() and core.N_VMin(vx) == x.min()
    for got, terms in ((core.N_VWrmsNorm(vx, vw), (x * w) ** 2),
                       (core.N_VWrmsNormMask(vx, vw, vi), (x * w) ** 2 * idv)):
        assert _close(got * got * n, terms) or abs(got * got * n / math.fsum(terms) - 1) <= (2 * n + 4) * 2.0 ** -53
    d = (C.c_double * 3)()
    assert core.N_VDotProdMulti(3, vx, vec_array([vx, vy, vw]), d) == 0
    assert all(_close(d[k], x * t) for k, t in enumerate((x, y, w)))
    # what is not finite comes through a result slot like any value
    x[n // 2] = np.nan
    vn = gpu_vec(ctx, x)
    assert math.isnan(core.N_VDotProd(vn, vy))
    x[n // 2] = np.inf
    vf = gpu_vec(ctx, x)
    assert core.N_VL1Norm(vf) == math.inf and core.N_VMaxNorm(vf) == math.inf
    for v in (vx, vy, vw, vz, vi, vn, vf):
        core.N_VDestroy(v)


def test_reduction_longer_than_the_watch(ctx):
    """Sequential order: one lane adds four million terms, far longer than the
    host watches the slot before it synchronises."""
    core, hip = _lib.core(), _lib.hip()
    n = 4000001
    x = np.random.default_rng(3).standard_normal(n)
    v = gpu_vec(ctx, x)
    assert hip.N_VSetReductionOrder_Mi355(v, 1) == 0
    want = np.cumsum(np.abs(x))[-1]  # left to right
    for _ in range(2):
        assert core.N_VL1Norm(v) == want
    core.N_VDestroy(v)


@pytest.mark.parametrize("k", [1, 8, 11, 12, 13, 23, 24, 25, 30])
def test_gram_schmidt_passes(ctx, k):
    core, hip = _lib.core(), _lib.hip()
    n = 70001
    rng = np.random.default_rng(k)
    q = np.linalg.qr(rng.standard_normal((n, k)))[0].T.copy()
    w = rng.standard_normal(n)
    vs = [gpu_vec(ctx, a) for a in q] + [gpu_vec(ctx, w)]
    tmp = [gpu_vec(ctx, np.zeros(n)) for _ in range(k + 1)]
    h = np.zeros((k + 1, k))
    PD = C.POINTER(C.c_double)
    rows = (PD * (k + 1))(*[C.cast(h[i].ctypes.data, PD) for i in range(k + 1)])
    norm, stemp = C.c_double(), (C.c_double * (k + 2))()
    assert hip.SUNAMD_ClassicalGS_Mi355(vec_array(vs), rows, k, k, C.byref(norm), stemp,
                                        vec_array(tmp)) == 0
    assert all(_close(h[i, k - 1], q[i] * w) for i in range(k))
    z = w.copy()
    for i in range(k):
        z = z + -h[i, k - 1] * q[i]
    assert np.array_equal(gpu_get(vs[-1]), z)
    assert abs(norm.value / np.linalg.norm(z) - 1) <= n * 2.0 ** -53
    for v in vs + tmp:
        core.N_VDestroy(v)


@pytest.mark.parametrize("with_cnrm", [False, True])
@pytest.mark.parametrize("n", EDGES)
def test_newton_update_equals_the_single_ops(ctx, n, with_cnrm):
    core, fn = _lib.core(), _lib.hip().cvNewtonUpdate_fused_Mi355
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p] * 5 + [C.POINTER(C.c_double)] * 2
    rng = np.random.default_rng(n)
    d, z, c = (rng.standard_normal(n) for _ in range(3))
    w = rng.uniform(0.5, 2, n)
    vd, vw, vz, vc, vy, ref_y = (gpu_vec(ctx, a) for a in (d, w, z, c, np.zeros(n), np.zeros(n)))
    dn, cn = C.c_double(-1.0), C.c_double(-1.0)
    assert fn(vd, vw, vz, vc, vy, C.byref(dn), C.byref(cn) if with_cnrm else None) == 0
    ref_c = gpu_vec(ctx, c)
    core.N_VLinearSum(1.0, ref_c, 1.0, vd, ref_c)
    core.N_VLinearSum(1.0, vz, 1.0, ref_c, ref_y)
    assert np.array_equal(gpu_get(vc), gpu_get(ref_c)) and np.array_equal(gpu_get(vy), gpu_get(ref_y))
    assert dn.value == core.N_VWrmsNorm(vd, vw)
    assert cn.value == (core.N_VWrmsNorm(ref_c, vw) if with_cnrm else -1.0)
    short = gpu_vec(ctx, np.zeros(n + 1))
    assert fn(vd, vw, vz, vc, short, C.byref(dn), None) == -1  # another length: nothing done
    assert fn(vd, vw, vz, vc, vz, C.byref(dn), None) == -1     # y is zn0
    assert np.array_equal(gpu_get(vc), gpu_get(ref_c))
    for v in (vd, vw, vz, vc, vy, ref_y, ref_c, short):
        core.N_VDestroy(v)


@pytest.mark.parametrize("q", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n", [1, 2, 2047, 2048, 2051, 300001])
def test_predictor_with_the_newton_start(ctx, n, q):
    core, hip = _lib.core(), _lib.hip()
    plain, start = hip.cvPredict_fused_Mi355, hip.cvPredictStart_fused_Mi355
    plain.restype = start.restype = C.c_int
    rng = np.random.default_rng(n + q)
    z = rng.standard_normal((q + 1, n))
    z[0, -1], z[1:, -1] = -0.0, -0.0  # -0 + 0 is +0 in y, and stays -0 in zn
    a, b = ([gpu_vec(ctx, r) for r in z] for _ in range(2))
    acor, y, ref = (gpu_vec(ctx, rng.standard_normal(n)) for _ in range(3))
    zero = gpu_vec(ctx, np.zeros(n))
    assert plain(q, vec_array(a)) == 0
    core.N_VLinearSum(1.0, a[0], 1.0, zero, ref)
    assert start(q, vec_array(b), C.c_void_p(acor), C.c_void_p(y)) == 0
    bits = lambda v: gpu_get(v).view(np.int64)  # noqa: E731
    assert all(np.array_equal(bits(u), bits(v)) for u, v in zip(a, b))
    assert np.array_equal(bits(y), bits(ref)) and not bits(acor).any()
    short = gpu_vec(ctx, np.zeros(n + 1))
    for bad in ((acor, short), (b[1], y), (acor, b[0]), (y, y)):
        assert start(q, vec_array(b), *map(C.c_void_p, bad)) == -1
    assert all(np.array_equal(bits(u), bits(v)) for u, v in zip(a, b))
    for v in (*a, *b, acor, y, ref, zero, short):
        core.N_VDestroy(v)


@pytest.mark.parametrize("n", EDGES)
def test_error_weights_with_the_norm(ctx, n):
    core, fn = _lib.core(), _lib.hip().cvEwtSetSSNorm_fused_Mi355
    fn.restype = C.c_int
    fn.argtypes = [C.c_double] * 2 + [C.c_void_p] * 3 + [C.POINTER(C.c_double)]
    x = np.random.default_rng(n).standard_normal(n)
    vx, vt, vw = (gpu_vec(ctx, a) for a in (x, np.zeros(n), np.zeros(n)))
    nrm = C.c_double(-1.0)
    assert fn(1e-5, 1e-9, vx, vt, vw, C.byref(nrm)) == 0
    t = 1e-5 * np.abs(x) + 1e-9
    assert np.array_equal(gpu_get(vt), t) and np.array_equal(gpu_get(vw), 1.0 / t)
    assert nrm.value == core.N_VWrmsNorm(vx, vw)
    assert fn(1e-5, 1e-9, vx, vx, vw, C.byref(nrm)) == -1
    for v in (vx, vt, vw):
        core.N_VDestroy(v)


@pytest.mark.parametrize("shared", ["ycor=delta", "ycor=ewt", "ycor=zn0", "y=delta", "y=ewt", "y=zn0",
                                    "y=ycor"])
def test_newton_update_declines_shared_outputs(ctx, shared):
    """N_VLinearSum into a vector that a later call of the sequence reads gives
    other values than one pass: such calls are declined and touch nothing."""
    core, fn = _lib.core(), _lib.hip().cvNewtonUpdate_fused_Mi355
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p] * 5 + [C.POINTER(C.c_double)] * 2
    n = 1001
    names = ("delta", "ewt", "zn0", "ycor", "y")
    vals = dict(zip(names, np.random.default_rng(5).uniform(0.5, 2, (5, n))))
    v = {k: gpu_vec(ctx, vals[k]) for k in names}
    out, other = shared.split("=")
    args = [v[other if k == out else k] for k in names]
    dn, cn = C.c_double(-1.0), C.c_double(-1.0)
    assert fn(*args, C.byref(dn), C.byref(cn)) == -1
    assert (dn.value, cn.value) == (-1.0, -1.0)
    assert all(np.array_equal(gpu_get(v[k]), vals[k]) for k in names)
    for k in names:
        core.N_VDestroy(v[k])
