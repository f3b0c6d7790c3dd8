"""SUNNonlinSol_NewtonSetUpdateInConvTest (no reference counterpart), on the CPU
with the serial vector: with the option on, the Newton solver leaves ycor +=
delta to its convergence test.  A test that makes that sum sees the iterates of
the plain loop bit for bit, through a restart from a cleared correction (a
recoverable failure with stale Jacobian data) as well."""
import ctypes as C

import numpy as np
import pytest

from sundials_amd import _lib
from test_newton_negated_host import (A, C0, CTestFn, LSolveFn, SUN_ERR_ARG_INCOMPATIBLE,
                                      SUN_NLS_CONTINUE, SysFn, _arr, libs)  # noqa: F401

LSetupFn = C.CFUNCTYPE(C.c_int, C.c_int, C.c_void_p, C.c_void_p)


def _run(core, orc, in_test, fail_at):
    ctx = _lib.new_context()
    y0, ycor, w = (orc.N_VNew_Serial(3, ctx) for _ in range(3))
    _arr(core, y0)[:] = [0.3, -0.7, 0.2]
    _arr(core, ycor)[:] = 0.0
    _arr(core, w)[:] = 1.0
    seen, calls = [], [0]

    def sys(yc, F, mem):
        y = _arr(core, y0) + _arr(core, yc)
        _arr(core, F)[:] = A @ y + 0.1 * y ** 3 - C0
        return 0

    def lsolve(b, mem):
        _arr(core, b)[:] = np.linalg.solve(A, _arr(core, b))
        return 0

    def ctest(nls, yc, dl, tol, ewt, data):
        if in_test:
            _arr(core, yc)[:] += _arr(core, dl)
        seen.append(_arr(core, yc).copy())
        calls[0] += 1
        if calls[0] == fail_at:
            return 902  # a recoverable failure
        nrm = float(np.sqrt(np.mean(_arr(core, dl) ** 2)))
        return 0 if nrm < tol else SUN_NLS_CONTINUE

    core.SUNNonlinSolSetLSetupFn.restype = C.c_int
    core.SUNNonlinSolSetLSetupFn.argtypes = [C.c_void_p, LSetupFn]
    cbs = (SysFn(sys), LSolveFn(lsolve), CTestFn(ctest), LSetupFn(lambda jbad, jcur, mem: 0))
    NLS = core.SUNNonlinSol_Newton(y0, ctx)
    assert core.SUNNonlinSolSetSysFn(NLS, cbs[0]) == 0
    assert core.SUNNonlinSolSetLSolveFn(NLS, cbs[1]) == 0
    assert core.SUNNonlinSolSetConvTestFn(NLS, cbs[2], None) == 0
    assert core.SUNNonlinSolSetLSetupFn(NLS, cbs[3]) == 0
    assert core.SUNNonlinSolSetMaxIters(NLS, 12) == 0
    assert core.SUNNonlinSolInitialize(NLS) == 0
    if in_test:
        assert core.SUNNonlinSol_NewtonSetUpdateInConvTest(C.c_void_p(NLS), 1) == 0
    rc = core.SUNNonlinSolSolve(NLS, y0, ycor, w, 1e-12, 0, None)
    core.SUNNonlinSolFree(NLS)
    for v in (y0, ycor, w):
        core.N_VDestroy(v)
    _lib.free_context(ctx)
    return rc, seen


@pytest.mark.parametrize("fail_at", [0, 1, 2])
def test_same_iterates(libs, fail_at):  # noqa: F811
    core, orc = libs
    rc_ref, ref = _run(core, orc, False, fail_at)
    rc_upd, upd = _run(core, orc, True, fail_at)
    assert rc_ref == rc_upd == 0 and len(ref) == len(upd) >= 3
    assert all(np.array_equal(a, b) for a, b in zip(ref, upd))
    assert core.SUNNonlinSol_NewtonSetUpdateInConvTest(None, 1) == SUN_ERR_ARG_INCOMPATIBLE
