"""CVODE's fused passes and the state of a step they share: the predictor that
also starts the Newton iteration, the update that also forms y, and what has to
void them -- an initial-correction callback (which may decline, propose zero,
propose something, or do these in turn), the fused mode switched on and off
between outputs, and a Newton solver attached by the program.  Each run equals
the run without fused kernels bit for bit at every output, in every counter."""
import ctypes as C

import numpy as np
import pytest

from sundials_amd import _lib
from helpers import gpu_get, gpu_vec

pytestmark = pytest.mark.gpu

CV_BDF, CV_NORMAL = 2, 1
P, D, I = C.c_void_p, C.c_double, C.c_int  # noqa: E741
InitFn = C.CFUNCTYPE(I, D, D, D, P, P, P)
TOUTS = (1e-3, 0.02, 0.05, 0.3, 1.0)


def _fn(lib, name, res, *args):
    return C.CFUNCTYPE(res, *args)((name, lib))


def _hook(core, kind):
    """kind -> CVInitialCorrectionFn body; a declining call leaves rubbish in
    the correction, which must not be used."""
    calls = [0]

    def decline(yp, ac):
        core.N_VScale(3.0, yp, ac)
        return 1

    def zero(yp, ac):
        core.N_VConst(0.0, ac)
        return 0

    def propose(yp, ac):
        core.N_VScale(1e-7, yp, ac)
        return 0

    bodies = {"declines": [decline], "zero": [zero], "proposes": [propose],
              "in turn": [decline, propose, zero, decline, decline, propose]}[kind]

    def call(t, h, gamma, yp, ac, user_data):
        calls[0] += 1
        return bodies[(calls[0] - 1) % len(bodies)](yp, ac)

    return call


def _run(m, R, ncells, order, fused, hook=None, own_solver=False):
    """fused: the mode before each output"""
    core, hip = _lib.core(), _lib.hip()
    ctx = _lib.new_context()
    p = core.SUNAMD_MassActionCreate(m, R, ncells, 1001, 0.2)
    n = m * ncells
    y = gpu_vec(ctx, np.ctypeslib.as_array(p.contents.y0, shape=(n,)).copy())
    assert hip.N_VSetReductionOrder_Mi355(y, order) == 0
    stream = hip.N_VGetStream_Mi355(y)
    dev = hip.SUNAMD_MassActionToDevice(p, C.c_void_p(stream))
    A = hip.SUNMatrix_Mi355BlockDense(ncells, m, stream, ctx)
    LS = hip.SUNLinSol_Mi355BlockLU(y, A, 0, ctx)
    cv = _fn(core, "CVodeCreate", P, I, P)(CV_BDF, ctx)
    assert dev and A and LS and cv
    rhs, jac = (C.cast(getattr(hip, s), P) for s in ("SUNAMD_MassActionRhsDev", "SUNAMD_MassActionJacDev"))
    assert _fn(core, "CVodeInit", I, P, P, D, P)(cv, rhs, 0.0, y) == 0
    assert _fn(core, "CVodeSStolerances", I, P, D, D)(cv, 1e-6, 1e-10) == 0
    assert _fn(core, "CVodeSetUserData", I, P, P)(cv, dev) == 0
    nls = None
    if own_solver:
        nls = _fn(core, "SUNNonlinSol_Newton", P, P, P)(y, ctx)
        assert _fn(core, "CVodeSetNonlinearSolver", I, P, P)(cv, nls) == 0
    assert _fn(core, "CVodeSetLinearSolver", I, P, P, P)(cv, LS, A) == 0
    assert _fn(core, "CVodeSetJacFn", I, P, P)(cv, jac) == 0
    assert _fn(core, "CVodeSetMaxNumSteps", I, P, C.c_long)(cv, 1000000) == 0
    cb = InitFn(_hook(core, hook)) if hook else None
    if hook:
        assert _fn(core, "CVodeSetInitialCorrectionFn", I, P, InitFn)(cv, cb) == 0
    step = _fn(core, "CVode", I, P, D, P, C.POINTER(D), I)
    mode = _fn(core, "CVodeSetUseIntegratorFusedKernels", I, P, I)
    out, t = [], D()
    for tout, on in zip(TOUTS, fused):
        assert mode(cv, on) == 0
        assert step(cv, tout, y, C.byref(t), CV_NORMAL) == 0
        cnt = []
        for name in ("NumSteps", "NumRhsEvals", "NumLinSolvSetups", "NumErrTestFails",
                     "NumNonlinSolvIters", "NumNonlinSolvConvFails", "NumInitialCorrectionsUsed"):
            v = C.c_long()
            assert _fn(core, "CVodeGet" + name, I, P, C.POINTER(C.c_long))(cv, C.byref(v)) == 0
            cnt.append(v.value)
        out.append((t.value, tuple(cnt), gpu_get(y)))
    launches = hip.N_VGetNumLaunches_Mi355(y)
    _fn(core, "CVodeFree", None, C.POINTER(P))(C.byref(P(cv)))
    if nls:
        _fn(core, "SUNNonlinSolFree", I, P)(nls)
    core.SUNLinSolFree(LS)
    core.SUNMatDestroy(A)
    hip.SUNAMD_MassActionDevFree(dev)
    core.N_VDestroy(y)
    core.SUNAMD_MassActionFree(p)
    _lib.free_context(ctx)
    return out, launches


def _same(got, ref):
    for (t, cnt, y), (tr, cr, yr) in zip(got, ref):
        assert cnt == cr and t == tr
        assert np.array_equal(y.view(np.int64), yr.view(np.int64))


ON, OFF = (1,) * 5, (0,) * 5


@pytest.mark.parametrize("order", [1, 0])  # sequential and tree sums
@pytest.mark.parametrize("m,R,ncells", [(8, 16, 65), (3, 4, 33)])
@pytest.mark.parametrize("hook", [None, "declines", "zero", "proposes", "in turn"])
def test_fused_mode_with_an_initial_correction(m, R, ncells, order, hook):
    ref, plain = _run(m, R, ncells, order, OFF, hook)
    got, fused = _run(m, R, ncells, order, ON, hook)
    _same(got, ref)
    assert fused < plain
    used = ref[-1][1][-1]
    assert (used > 0) == (hook in ("zero", "proposes", "in turn"))
    _same(_run(m, R, ncells, order, (1, 0, 1, 1, 0), hook)[0], ref)
    _same(_run(m, R, ncells, order, (0, 1, 0, 0, 1), hook)[0], ref)


def test_fused_mode_with_the_programs_own_solver():
    ref, _ = _run(8, 16, 65, 0, OFF, "in turn", own_solver=True)
    _same(_run(8, 16, 65, 0, (1, 1, 0, 1, 1), "in turn", own_solver=True)[0], ref)
    _same(_run(8, 16, 65, 0, ON, "in turn")[0], ref)
