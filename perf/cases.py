"""The work that programs built on this library have it do, as timed cases.

Each case is a dict of plain values; its "kind" is one of

  vector   the N_Vector ops of one BDF step (residual, Newton update, history
           update, error weights and norms)
  krylov   one Gram-Schmidt step of a Krylov solver on N_Vectors
  lu       Newton-matrix set-up and the solves with its factors on a
           block-diagonal matrix (batched LU)
  chem     mass-action right-hand side and block Jacobian of many cells
  bucket   independent stiff systems of one size in caller-owned buffers
  batch    an uneven batch of independent stiff systems, one integrator each
  coupled  all cells as one coupled BDF integration
  imex     ARKStep IMEX + SPGMR on the advection-diffusion-reaction problem
  mlp      training of the learned initial Newton iterate

Inputs come from the seed alone.  Whole integrations return their final
states; single steps return everything they compute.
"""
import ctypes as C
import math

import numpy as np
import torch

from sundials_amd import _lib

PD = C.POINTER(C.c_double)

# block sizes the coupled and per-system integrators take
SIZES = (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 16, 24, 32, 48, 64)
# the uneven batch: systems of these sizes in these shares
BATCH_M = (4, 8, 16, 24, 32, 48, 64)
BATCH_W = (0.30, 0.25, 0.15, 0.10, 0.10, 0.05, 0.05)
# BDF steps that one such system takes from t = 0 to 1 (rtol 1e-6), Newton
# iterations per step and steps per factorisation: for the flop counts
STEPS, NEWTON, PER_SETUP = 475, 1.37, 8.0


def listed():
    return [
        # 4096 cells x 8 species, one host-stepped BDF step of a small model:
        # launches and synchronisations count
        {"name": "vector_small", "kind": "vector", "n": 32768, "q": 3},
        # 2^20 cells x 32 species: the streaming range
        {"name": "vector_large", "kind": "vector", "n": 1 << 25, "q": 3},
        # one Arnoldi step of the 128^3 x 3 IMEX problem's SPGMR, half way
        # through a cycle of 20
        {"name": "krylov_cgs", "kind": "krylov", "n": 3 * 128 ** 3, "k": 10, "gs": "classical"},
        # Newton systems of 32-species cells as the fused CVODE mode calls the
        # solver (one-pass set-up, in-place solves)
        {"name": "lu_m32", "kind": "lu", "m": 32, "blocks": 1 << 18, "fp32": False,
         "fused": True, "solves": 4},
        # a mechanism of a size between the usual ones, single-precision
        # factors, through the matrix and solver calls a SUNDIALS program makes
        {"name": "lu_m21_fp32", "kind": "lu", "m": 21, "blocks": 50000, "fp32": True,
         "fused": False, "solves": 4},
        # right-hand side and Jacobian of 32-species cells
        {"name": "chem_m32", "kind": "chem", "m": 32, "R": 48, "cells": 1 << 18},
        # a host code's own small set of cells in buffers of its own: one
        # system's chain of dependent steps is what takes the time
        {"name": "bucket_small", "kind": "bucket", "m": 8, "R": 12, "cells": 64, "fp32": False},
        # the uneven batch in plain double precision
        {"name": "batch_fp64", "kind": "batch", "systems": 16384, "fp32": False},
        # the uneven batch of the benchmark in the product form
        # (single-precision Newton-matrix factors)
        {"name": "batch_fp32", "kind": "batch", "systems": 65536, "fp32": True},
        # 2^14 cells x 32 species as one integration, host-stepped with the
        # integrator's fused kernels
        {"name": "coupled_m32", "kind": "coupled", "m": 32, "cells": 1 << 14, "fp32": False,
         "device": False},
        # ARKStep IMEX, SPGMR with the device Gram-Schmidt step, on 128^3 cells
        {"name": "imex_128", "kind": "imex", "n": 128, "tf": 0.01, "fp32": False},
        # training of the initial iterate: Adam steps on logged pairs resident
        # on the device
        {"name": "mlp_train", "kind": "mlp", "rows": 32768, "batch": 1024, "steps": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("vector", "vector", "krylov", "lu", "lu", "lu", "chem", "chem", "bucket",
                       "batch", "coupled", "imex", "mlp"))
    if kind == "vector":
        return {"kind": kind, "n": _log_int(rng, 24, 1 << 25), "q": rng.randint(1, 5)}
    if kind == "krylov":
        k = rng.randint(1, 20)
        return {"kind": kind, "n": _log_int(rng, 1000, (3 * 128 ** 3 * 10) // max(k, 10)), "k": k,
                "gs": rng.choice(("classical", "modified"))}
    if kind == "lu":
        # any block size a SUNDIALS program may have, up to 512 MiB of blocks
        m = rng.randint(2, 64)
        blocks = _log_int(rng, 64, min(1 << 20, (1 << 29) // (8 * m * m)))
        return {"kind": kind, "m": m, "blocks": blocks, "fp32": rng.random() < 0.5,
                "fused": rng.random() < 0.5, "solves": rng.randint(1, 8)}
    if kind == "chem":
        m = rng.randint(2, 64)
        return {"kind": kind, "m": m, "R": max(1, int(round(1.5 * m))),
                "cells": _log_int(rng, 64, min(1 << 20, (1 << 30) // (8 * m * m)))}
    if kind == "bucket":
        m = rng.choice(SIZES[2:])
        return {"kind": kind, "m": m, "R": max(1, int(round(1.5 * m))),
                "cells": _log_int(rng, 16, 65536 // m), "fp32": rng.random() < 0.5}
    if kind == "batch":
        return {"kind": kind, "systems": _log_int(rng, 512, 16384), "fp32": rng.random() < 0.5}
    if kind == "coupled":
        m = rng.choice((3, 8, 16, 24, 32))
        return {"kind": kind, "m": m, "cells": _log_int(rng, 64, (1 << 18) // m),
                "fp32": rng.random() < 0.5, "device": rng.random() < 0.5}
    if kind == "imex":
        return {"kind": kind, "n": _log_int(rng, 16, 112), "tf": 0.01,
                "fp32": rng.random() < 0.5}
    batch = 16 * rng.randint(4, 128)
    return {"kind": "mlp", "rows": batch * rng.randint(4, 32), "batch": batch,
            "steps": rng.randint(4, 24)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _State:
    """What a program keeps between calls; `free` runs when it is dropped."""

    def __init__(self):
        self.free = []

    def __del__(self):
        for f in reversed(self.free):
            f()


def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _chemistry(m, R, cells, seed):
    """Reversible reactions a + b <-> c + d with log-uniform rates on
    [1e-2, 1e6], a lognormal factor per cell and rate, and a state per cell."""
    g = _gen(seed)
    idx = torch.randint(0, m, (R, 4), generator=g, device="cuda", dtype=torch.int32)
    k0 = 10.0 ** (8.0 * _rand(g, 2, 1, R) - 2.0)
    k = k0 * torch.exp(0.2 * _randn(g, 2, cells, R))
    y = 0.1 + 0.9 * _rand(g, cells, m)
    return idx, k[0].contiguous(), k[1].contiguous(), y / y.sum(1, keepdim=True)


def _stoichiometry(idx, m):
    """f = w F and J = p S with w the R net rates and p their 4R partials."""
    R = idx.shape[0]
    sign = (-1.0, -1.0, 1.0, 1.0)
    F = np.zeros((R, m))
    S = np.zeros((4 * R, m * m))
    for r, ix in enumerate(idx.cpu().numpy()):
        for t in range(4):
            F[r, ix[t]] += sign[t]
            for c in range(4):
                S[4 * r + c, ix[c] * m + ix[t]] += sign[t]
    return torch.from_numpy(F).cuda(), torch.from_numpy(S).cuda()


def _rhs_and_jacobian(idx, kf, kb, y):
    m = y.shape[1]
    ix = idx.long()
    F, S = _stoichiometry(idx, m)
    a, b, c, d = (y[:, ix[:, t]] for t in range(4))
    f = (kf * a * b - kb * c * d) @ F
    p = torch.stack((kf * b, kf * a, -(kb * d), -(kb * c)), dim=2).reshape(y.shape[0], -1)
    return f, p @ S


def _nvector(s, t):
    """An N_Vector on a device tensor's memory."""
    v = _lib.hip().N_VMake_Mi355(t.numel(), None, t.data_ptr(), s.ctx)
    if not v:
        raise RuntimeError("N_VMake_Mi355 failed")
    s.free.append(lambda: _lib.core().N_VDestroy(v))
    return v


def _context(s):
    s.ctx = _lib.new_context()
    s.free.append(lambda: _lib.free_context(s.ctx))


def _vecs(vs):
    return (C.c_void_p * len(vs))(*vs)


def _ok(rc, what):
    if rc != 0:
        raise RuntimeError("%s returned %s" % (what, rc))


def prepare(case, seed):
    s = _State()
    s.case = case
    s.core, s.hip = _lib.core(), _lib.hip()
    _PREPARE[case["kind"]](s, case, seed)
    # the library's streams do not wait for torch's
    torch.cuda.synchronize()
    return s


def run(state):
    return _RUN[state.case["kind"]](state, state.case)


# ---------------------------------------------------------------------------
# vector: one step's ops at order q
# ---------------------------------------------------------------------------
def _vector_inputs(case, seed):
    n, q, g = case["n"], case["q"], _gen(seed)
    y = _rand(g, n) / 8.0
    zn = [y] + [y * _randn(g, n) * 10.0 ** -j for j in range(1, q + 1)]
    acor, f = 1e-6 * _randn(g, n), _randn(g, n)
    coef = [float(v) for v in torch.rand(2 * (q + 1), generator=torch.Generator().manual_seed(int(seed)),
                                         dtype=torch.float64) + 0.1]
    return zn, acor, f, coef[:q + 1], coef[q + 1:]


def _prepare_vector(s, case, seed):
    n, q = case["n"], case["q"]
    _context(s)
    zn, acor, f, l, c = _vector_inputs(case, seed)
    s.out = {k: torch.zeros(n, dtype=torch.float64, device="cuda")
             for k in ("res", "corr", "y", "ewt", "comb")}
    s.out["zn"] = [torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(q + 1)]
    s.keep = (zn, acor, f)
    s.zn, s.acor, s.f = [_nvector(s, t) for t in zn], _nvector(s, acor), _nvector(s, f)
    s.o = {k: _nvector(s, t) for k, t in s.out.items() if k != "zn"}
    s.o["zn"] = [_nvector(s, t) for t in s.out["zn"]]
    s.l, s.c = (C.c_double * (q + 1))(*l), (C.c_double * (q + 1))(*c)
    s.znp, s.onp = _vecs(s.zn), _vecs(s.o["zn"])


def _run_vector(s, case):
    core, o, q1 = s.core, s.o, case["q"] + 1
    # error weights of the current state
    core.N_VAbs(s.zn[0], o["ewt"])
    core.N_VScale(1e-6, o["ewt"], o["ewt"])
    core.N_VAddConst(o["ewt"], 1e-10, o["ewt"])
    core.N_VInv(o["ewt"], o["ewt"])
    # nonlinear residual zn[1] / l1 + acor - gamma f
    core.N_VLinearSum(0.8, s.zn[1], 1.0, s.acor, o["res"])
    core.N_VLinearSum(-1e-3, s.f, 1.0, o["res"], o["res"])
    rnorm = core.N_VWrmsNorm(o["res"], o["ewt"])
    # Newton update and the predicted state plus the correction
    core.N_VLinearSum(1.0, s.acor, 1.0, o["res"], o["corr"])
    core.N_VLinearSum(1.0, s.zn[0], 1.0, o["corr"], o["y"])
    dsm = core.N_VWrmsNorm(o["corr"], o["ewt"])
    # history update and interpolation of the new history
    _ok(core.N_VScaleAddMulti(q1, s.l, o["corr"], s.znp, s.onp), "N_VScaleAddMulti")
    _ok(core.N_VLinearCombination(q1, s.c, s.onp, o["comb"]), "N_VLinearCombination")
    big = core.N_VMaxNorm(o["comb"])
    return {"vectors": s.out, "norms": np.array([rnorm, dsm, big])}


def _exact_vector(case, seed):
    zn, acor, f, l, c = _vector_inputs(case, seed)
    ewt = 1.0 / (1e-6 * zn[0].abs() + 1e-10)
    res = 0.8 * zn[1] + acor - 1e-3 * f
    corr = acor + res
    new = [l[j] * corr + zn[j] for j in range(len(zn))]
    comb = sum(c[j] * new[j] for j in range(len(zn)))
    rms = lambda v: float((v * ewt).square().mean().sqrt())  # noqa: E731
    return {"vectors": {"res": res, "corr": corr, "y": zn[0] + corr, "ewt": ewt, "comb": comb,
                        "zn": new},
            "norms": np.array([rms(res), rms(corr), float(comb.abs().max())])}


# ---------------------------------------------------------------------------
# krylov: v_k made orthogonal to v_0 .. v_{k-1}
# ---------------------------------------------------------------------------
def _krylov_inputs(case, seed):
    n, k, g = case["n"], case["k"], _gen(seed)
    basis = []
    for _ in range(k):
        v = _randn(g, n)
        for _ in range(2):
            for u in basis:
                v -= torch.dot(u, v) * u
        basis.append(v / v.norm())
    w = _randn(g, n)
    w /= w.norm()
    for u, c in zip(basis, _randn(g, k).cpu().tolist()):
        w += c * u
    return basis, w


def _prepare_krylov(s, case, seed):
    n, k = case["n"], case["k"]
    _context(s)
    basis, w = _krylov_inputs(case, seed)
    s.vk = torch.zeros_like(w)
    temps = [torch.zeros_like(w) for _ in range(k + 1)] if case["gs"] == "classical" else []
    s.keep = (basis, w, temps)
    s.w = _nvector(s, w)
    vs = [_nvector(s, t) for t in basis] + [_nvector(s, s.vk)]
    s.last, s.v = vs[-1], _vecs(vs)
    s.h = np.zeros((k + 1, k))
    s.rows = (PD * (k + 1))(*[C.cast(s.h[i].ctypes.data, PD) for i in range(k + 1)])
    s.norm, s.stemp = C.c_double(), (C.c_double * (k + 2))()
    s.vtemp = _vecs([_nvector(s, t) for t in temps]) if temps else None


def _run_krylov(s, case):
    k = case["k"]
    s.core.N_VScale(1.0, s.w, s.last)
    if case["gs"] == "classical":
        _ok(s.hip.SUNAMD_ClassicalGS_Mi355(s.v, s.rows, k, k, C.byref(s.norm), s.stemp, s.vtemp),
            "SUNAMD_ClassicalGS_Mi355")
    else:
        _ok(s.core.SUNModifiedGS(s.v, s.rows, k, k, C.byref(s.norm)), "SUNModifiedGS")
    return {"v": s.vk, "h": s.h[:k, k - 1].copy(), "norm": s.norm.value}


def _exact_krylov(case, seed):
    basis, w = _krylov_inputs(case, seed)
    h = [float(torch.dot(u, w)) for u in basis]
    v = w.clone()
    for u, c in zip(basis, h):
        v -= c * u
    return {"v": v, "h": np.array(h), "norm": float(v.norm())}


# ---------------------------------------------------------------------------
# lu: I - gamma J from the saved Jacobian, factored once, solved several times
# ---------------------------------------------------------------------------
# a step size early in an integration: rates times GAMMA reach about 10
GAMMA, SCALE = 1e-4, 0.9


def _lu_inputs(case, seed):
    m, nb = case["m"], case["blocks"]
    idx, kf, kb, y = _chemistry(m, max(1, int(round(1.5 * m))), nb, seed)
    J = _rhs_and_jacobian(idx, kf, kb, y)[1]
    g = _gen(seed + 977)
    return J, [1e-3 * _randn(g, nb * m) for _ in range(case["solves"])]


def _prepare_lu(s, case, seed):
    m, nb = case["m"], case["blocks"]
    core, hip = s.core, s.hip
    _context(s)
    J, b = _lu_inputs(case, seed)
    s.rhs, s.x = b, [torch.zeros_like(t) for t in b]
    s.b = [_nvector(s, t) for t in s.rhs]
    s.xv = [_nvector(s, t) for t in s.x]
    stream = hip.N_VGetStream_Mi355(s.b[0])
    s.A = hip.SUNMatrix_Mi355BlockDense(nb, m, stream, s.ctx)
    s.J = hip.SUNMatrix_Mi355BlockDense(nb, m, stream, s.ctx)
    if not s.A or not s.J:
        raise RuntimeError("SUNMatrix_Mi355BlockDense failed")
    s.free += [lambda: core.SUNMatDestroy(s.A), lambda: core.SUNMatDestroy(s.J)]
    # the Jacobian's blocks go where a user's Jacobian function writes them
    torch.cuda.synchronize()
    dst = hip.N_VMake_Mi355(J.numel(), None, hip.SUNMatrix_Mi355BlockDense_DeviceData(s.J), s.ctx)
    core.N_VScale(1.0, _nvector(s, J), dst)
    _ok(hip.N_VSynchronize_Mi355(dst), "N_VSynchronize_Mi355")
    core.N_VDestroy(dst)
    s.S = hip.SUNLinSol_Mi355BlockLU(s.b[0], s.A, 1 if case["fp32"] else 0, s.ctx)
    if not s.S:
        raise RuntimeError("SUNLinSol_Mi355BlockLU failed")
    s.free.append(lambda: core.SUNLinSolFree(s.S))
    core.SUNLinSolInitialize(s.S)


def _run_lu(s, case):
    core, hip = s.core, s.hip
    declined = -9998
    rc = declined
    if case["fused"]:
        rc = hip.SUNLinSol_Mi355BlockLUSetupScaled(s.S, s.A, s.J, -GAMMA, 0)
    # a solver declines the one-pass call where it has none (negative): the
    # three calls follow, as in the integrator
    if rc < 0:
        _ok(core.SUNMatCopy(s.J, s.A), "SUNMatCopy")
        _ok(core.SUNMatScaleAddI(-GAMMA, s.A), "SUNMatScaleAddI")
        rc = core.SUNLinSolSetup(s.S, s.A)
    _ok(rc, "linear solver setup")
    for b, x in zip(s.b, s.xv):
        rc = declined
        if case["fused"]:
            core.N_VScale(1.0, b, x)
            rc = hip.SUNLinSol_Mi355BlockLUSolveScaled(s.S, s.A, x, SCALE)
        if rc < 0:
            core.N_VConst(0.0, x)
            _ok(core.SUNLinSolSolve(s.S, s.A, x, b, 0.0), "SUNLinSolSolve")
            core.N_VScale(SCALE, x, x)
    return s.x


def _exact_lu(case, seed):
    m, nb = case["m"], case["blocks"]
    J, b = _lu_inputs(case, seed)
    A = torch.eye(m, dtype=torch.float64, device="cuda") - GAMMA * J.reshape(nb, m, m).transpose(1, 2)
    x = torch.linalg.solve(A.contiguous(), torch.stack([t.reshape(nb, m) for t in b], dim=2))
    return [SCALE * x[:, :, j].reshape(-1) for j in range(case["solves"])]


# ---------------------------------------------------------------------------
# chem: f(y) and J(y) of every cell
# ---------------------------------------------------------------------------
def _prepare_chem(s, case, seed):
    m, R, cells = case["m"], case["R"], case["cells"]
    idx, kf, kb, s.y = _chemistry(m, R, cells, seed)
    host = [np.ascontiguousarray(t.cpu().numpy()) for t in (idx, kf, kb, s.y)]
    ptr = lambda a, t: a.ctypes.data_as(C.POINTER(t))  # noqa: E731
    p = _lib.MassAction(m=m, R=R, ncells=cells, seed=0, sigma=0.2, idx=ptr(host[0], C.c_int),
                        kf=ptr(host[1], C.c_double), kb=ptr(host[2], C.c_double),
                        y0=ptr(host[3], C.c_double))
    s.d = s.hip.SUNAMD_MassActionToDevice(C.byref(p), None)
    if not s.d:
        raise RuntimeError("SUNAMD_MassActionToDevice failed")
    s.free.append(lambda: s.hip.SUNAMD_MassActionDevFree(s.d))
    s.f = torch.zeros(cells, m, dtype=torch.float64, device="cuda")
    s.J = torch.zeros(cells, m * m, dtype=torch.float64, device="cuda")


def _run_chem(s, case):
    _ok(s.hip.SUNAMD_MassActionRhsDevArrays(s.d, s.y.data_ptr(), s.f.data_ptr()), "rhs")
    _ok(s.hip.SUNAMD_MassActionJacDevArrays(s.d, s.y.data_ptr(), s.J.data_ptr()), "jacobian")
    return {"f": s.f, "J": s.J}


def _exact_chem(case, seed):
    idx, kf, kb, y = _chemistry(case["m"], case["R"], case["cells"], seed)
    f, J = _rhs_and_jacobian(idx, kf, kb, y)
    return {"f": f, "J": J}


# ---------------------------------------------------------------------------
# bucket: systems of one size in the caller's buffers
# ---------------------------------------------------------------------------
def _prepare_bucket(s, case, seed):
    m, cells = case["m"], case["cells"]
    s.idx, s.kf, s.kb, s.y = _chemistry(m, case["R"], cells, seed)
    s.out = torch.zeros(cells, m, dtype=torch.float64, device="cuda")
    s.counters = torch.zeros(cells, _lib.BS_COUNT, dtype=torch.int64, device="cuda")


def _run_bucket(s, case):
    _ok(s.hip.SUNAMD_BatchedBDFSolveBucketNoAlloc(
        case["m"], case["R"], case["cells"], s.idx.data_ptr(), s.kf.data_ptr(), s.kb.data_ptr(),
        s.y.data_ptr(), 1e-6, 1e-10, 1.0, 100000, 1 if case["fp32"] else 0, s.out.data_ptr(),
        s.counters.data_ptr(), torch.cuda.current_stream().cuda_stream), "bucket solve")
    # the counters of the double-precision form are the reference integrator's;
    # those of the single-precision factors follow their rounding
    return {"y": s.out} if case["fp32"] else {"y": s.out, "counters": s.counters}


# ---------------------------------------------------------------------------
# batch: the uneven batch, results in system order on the host
# ---------------------------------------------------------------------------
def _prepare_batch(s, case, seed):
    nb = len(BATCH_M)
    b = s.core.SUNAMD_BatchCreate(case["systems"], seed, nb, (C.c_int * nb)(*BATCH_M),
                                  (C.c_double * nb)(*BATCH_W), 1.5, 0.2)
    if not b:
        raise RuntimeError("SUNAMD_BatchCreate failed")
    s.nsys = b.contents.nsys
    # room for any seed's sizes (16.8 species per system on average)
    s.room = int(17 * s.nsys + 160 * math.sqrt(s.nsys))
    if b.contents.ytotal > s.room:
        raise RuntimeError("batch larger than its result buffer")
    s.B = s.hip.SUNAMD_BatchedBDFCreate(b, 1e-6, 1e-10, 1 if case["fp32"] else 0)
    buckets = b.contents.nbuckets
    s.core.SUNAMD_BatchFree(b)
    if not s.B:
        raise RuntimeError("SUNAMD_BatchedBDFCreate failed")
    s.free.append(lambda: s.hip.SUNAMD_BatchedBDFFree(s.B))
    # the launch settings a calibration run settles on
    waves = 3 if case["fp32"] else 2
    _ok(s.hip.SUNAMD_BatchedBDFSetMaxNumSteps(s.B, 100000), "max steps")
    _ok(s.hip.SUNAMD_BatchedBDFSetOccupancy(s.B, (C.c_int * buckets)(*([waves] * buckets))),
        "occupancy")


def _run_batch(s, case):
    wall = C.c_double()
    _ok(s.hip.SUNAMD_BatchedBDFRun(s.B, 1.0, C.byref(wall)), "batched run")
    y = np.zeros(s.room)
    if case["fp32"]:
        _ok(s.hip.SUNAMD_BatchedBDFGetResults(s.B, y.ctypes.data_as(PD), None), "batched results")
        return {"y": y}
    counters = np.empty((s.nsys, _lib.BS_COUNT), dtype=np.int64)
    _ok(s.hip.SUNAMD_BatchedBDFGetResults(s.B, y.ctypes.data_as(PD),
                                          counters.ctypes.data_as(C.POINTER(C.c_long))),
        "batched results")
    return {"y": y, "counters": counters}


# ---------------------------------------------------------------------------
# coupled: one integrator for all cells
# ---------------------------------------------------------------------------
def _prepare_coupled(s, case, seed):
    m, cells = case["m"], case["cells"]
    p = s.core.SUNAMD_MassActionCreate(m, max(1, int(round(1.5 * m))), cells, seed, 0.2)
    if not p:
        raise RuntimeError("SUNAMD_MassActionCreate failed")
    s.r = s.hip.SUNAMD_CoupledCreate_Mi355(p, 1e-6, 1e-10, 1 if case["fp32"] else 0, 0)
    s.core.SUNAMD_MassActionFree(p)
    if not s.r:
        raise RuntimeError("SUNAMD_CoupledCreate_Mi355 failed")
    s.free.append(lambda: s.hip.SUNAMD_CoupledFree_Mi355(s.r))
    if case["device"]:
        _ok(s.hip.SUNAMD_CoupledSetDeviceStepping_Mi355(s.r, 1), "device stepping")
    else:
        _ok(s.hip.SUNAMD_CoupledSetFusedKernels_Mi355(s.r, 1), "fused kernels")


def _run_coupled(s, case):
    st = _lib.SolveStats()
    _ok(s.hip.SUNAMD_CoupledRun_Mi355(s.r, 1.0, C.byref(st)), "coupled run")
    y = np.empty(case["cells"] * case["m"])
    _ok(s.hip.SUNAMD_CoupledGetState_Mi355(s.r, y.ctypes.data_as(PD)), "coupled state")
    return y


# ---------------------------------------------------------------------------
# imex: one ARKStep solve, integrator and Krylov workspace included
# ---------------------------------------------------------------------------
def _prepare_imex(s, case, seed):
    s.p = s.core.SUNAMD_AdrCreate(case["n"], seed)
    if not s.p:
        raise RuntimeError("SUNAMD_AdrCreate failed")
    s.free.append(lambda: s.core.SUNAMD_AdrFree(s.p))
    s.o = _lib.AdrOptions(1e-6, 1e-10, case["tf"], 20, 2, 0, 0, 1 if case["fp32"] else 0, 1000000)


def _run_imex(s, case):
    st, y = np.zeros(_lib.ADR_STATS), np.empty(3 * case["n"] ** 3)
    _ok(s.hip.SUNAMD_AdrSolve_Mi355(s.p, C.byref(s.o), st.ctypes.data_as(PD), y.ctypes.data_as(PD)),
        "imex solve")
    return y


# ---------------------------------------------------------------------------
# mlp: Adam steps on logged pairs
# ---------------------------------------------------------------------------
NPARAM = 128 * 144 + 128 + 128 * 128 + 128 + 64 * 128 + 64
MLP_SEED, LR = 17, 1e-3


def _mlp_inputs(case, seed):
    """Rows as the batched integrator logs them: log10 of the predicted state,
    of gamma and of the rate sums, each / 10; corrections in error-weight
    units; the species mask."""
    n, g = case["rows"], _gen(seed)
    f32 = lambda *sh: torch.rand(*sh, generator=g, device="cuda", dtype=torch.float32)  # noqa: E731
    sizes = torch.tensor(BATCH_M, device="cuda")
    m = sizes[torch.randint(0, len(BATCH_M), (n,), generator=g, device="cuda")]
    mask = (torch.arange(64, device="cuda")[None, :] < m[:, None]).float()
    x = torch.zeros(n, 144, device="cuda")
    x[:, :64] = -0.6 * f32(n, 64) * mask
    x[:, 64] = -0.8 * f32(n)
    x[:, 65:129] = 0.7 * f32(n, 64) * mask
    t = 5.0 * torch.randn(n, 64, generator=g, device="cuda") * mask
    t += 20.0 * (x[:, :64] + x[:, 65:129]) * mask
    return x, t.contiguous(), mask.contiguous()


def _prepare_mlp(s, case, seed):
    s.x, s.t, s.mask = _mlp_inputs(case, seed)
    s.M = s.hip.SUNAMD_MLPCreate(MLP_SEED, case["batch"])
    if not s.M:
        raise RuntimeError("SUNAMD_MLPCreate failed")
    s.free.append(lambda: s.hip.SUNAMD_MLPFree(s.M))


def _run_mlp(s, case):
    loss, params = C.c_float(), np.empty(NPARAM, dtype=np.float32)
    _ok(s.hip.SUNAMD_MLPTrain(s.M, s.x.data_ptr(), s.t.data_ptr(), s.mask.data_ptr(), case["rows"],
                              case["batch"], case["steps"], LR, C.byref(loss)), "training")
    _ok(s.hip.SUNAMD_MLPGetParams(s.M, params.ctypes.data_as(C.POINTER(C.c_float))), "parameters")
    return {"params": params, "loss": loss.value}


def _initial_params():
    """The seeded initial weights (SplitMix64, uniform +-scale sqrt(6 / inputs))."""
    mask = (1 << 64) - 1
    st = (MLP_SEED * 0x9E3779B97F4A7C15 + 0x632BE59BD9B4E5F) & mask
    # state k's output depends on st + k * step alone
    count = 128 * 129 + 128 * 128 + 64 * 128
    with np.errstate(over="ignore"):
        z = np.uint64(st) + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, count + 1, dtype=np.uint64)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z ^= z >> np.uint64(31)
    u = 2.0 * ((z >> np.uint64(11)).astype(np.float64) / 9007199254740992.0) - 1.0
    out, at = [], 0
    for rows, used, cols, scale in ((128, 129, 144, 1.0), (128, 128, 128, 1.0), (64, 128, 128, 0.1)):
        w = np.zeros((rows, cols), dtype=np.float32)
        w[:, :used] = u[at:at + rows * used].reshape(rows, used) * (scale * math.sqrt(6.0 / used))
        at += rows * used
        out += [w, np.zeros(rows, dtype=np.float32)]
    return out


def _exact_mlp(case, seed):
    x, t, mask = (v.double() for v in _mlp_inputs(case, seed))
    p = [torch.from_numpy(w).cuda().double().requires_grad_() for w in _initial_params()]
    m1, m2 = [torch.zeros_like(w) for w in p], [torch.zeros_like(w) for w in p]
    silu = torch.nn.functional.silu
    losses = []
    for k in range(case["steps"]):
        at = (k * case["batch"]) % case["rows"]
        at = min(at, case["rows"] - case["batch"])
        rows = slice(at, at + case["batch"])
        a = silu(x[rows] @ p[0].T + p[1])
        a = silu(a @ p[2].T + p[3])
        d = (a @ p[4].T + p[5] - t[rows]) * mask[rows]
        loss = d.square().sum() / mask[rows].sum()
        losses.append(float(loss))
        with torch.no_grad():
            for w, g, u, v in zip(p, torch.autograd.grad(loss, p), m1, m2):
                u.mul_(0.9).add_(g, alpha=0.1)
                v.mul_(0.999).add_(g * g, alpha=0.001)
                w -= LR * (u / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    flat = torch.cat([w.detach().reshape(-1) for w in p])
    return {"params": flat, "loss": float(np.mean(losses[-10:]))}


_PREPARE = {"vector": _prepare_vector, "krylov": _prepare_krylov, "lu": _prepare_lu,
            "chem": _prepare_chem, "bucket": _prepare_bucket, "batch": _prepare_batch,
            "coupled": _prepare_coupled, "imex": _prepare_imex, "mlp": _prepare_mlp}
_RUN = {"vector": _run_vector, "krylov": _run_krylov, "lu": _run_lu, "chem": _run_chem,
        "bucket": _run_bucket, "batch": _run_batch, "coupled": _run_coupled, "imex": _run_imex,
        "mlp": _run_mlp}
_EXACT = {"vector": _exact_vector, "krylov": _exact_krylov, "lu": _exact_lu, "chem": _exact_chem,
          "mlp": _exact_mlp}


def exact(case, seed):
    """None for whole integrations: a reference far inside their tolerance
    (rtol 1e-6 on stiff systems) takes plain torch minutes."""
    f = _EXACT.get(case["kind"])
    return f(case, seed) if f else None


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far a correct one may be off
# ---------------------------------------------------------------------------
def _bdf_flops(m, R):
    """One system's integration: factorisations, solves, right-hand sides."""
    return STEPS * ((2.0 / 3.0 * m ** 3 + 24.0 * R) / PER_SETUP + NEWTON * (2.0 * m * m + 20.0 * R))


def work(case):
    kind = case["kind"]
    if kind == "vector":
        n, q = case["n"], case["q"]
        # four unary ops, four sums, three norms, the two fused ops
        per = 4 * 16 + 4 * 24 + 2 * 16 + 8 + 8 * (2 * (q + 1) + 1) + 8 * (q + 2)
        return {"bytes": per * n, "flops": (4 + 4 * 3 + 3 * 3 + 4 * (q + 1)) * n}
    if kind == "krylov":
        n, k = case["n"], case["k"]
        # the copy of w; the basis for the projections and again for the
        # update that needs them, w read twice more and written
        return {"bytes": 8 * n * (2 + 2 * k + 3), "flops": (4 * k + 4) * n}
    if kind == "lu":
        m, nb, f = case["m"], case["blocks"], 4 if case["fp32"] else 8
        return {"bytes": nb * ((8 + f) * m * m + 4 * m + case["solves"] * (f * m * m + 20 * m)),
                "flops": nb * (2.0 / 3.0 * m ** 3 + 2 * m * m * case["solves"])}
    if kind == "chem":
        m, R, c = case["m"], case["R"], case["cells"]
        return {"bytes": 8 * c * (2 * (m + 2 * R) + m + m * m), "flops": c * (7 * R + 8 * R + 16 * R)}
    if kind == "bucket":
        m, R, c = case["m"], case["R"], case["cells"]
        return {"bytes": 8 * c * (2 * m + 2 * R + 10), "flops": c * _bdf_flops(m, R)}
    if kind == "batch":
        n = case["systems"]
        return {"bytes": n * sum(w * 8 * (2 * m + 3 * m + 10) for m, w in zip(BATCH_M, BATCH_W)),
                "flops": n * sum(w * _bdf_flops(m, 1.5 * m) for m, w in zip(BATCH_M, BATCH_W))}
    if kind == "coupled":
        # state, history, weights, correction, rates and factors move once per
        # Newton iteration: about 1300 steps
        m, c = case["m"], case["cells"]
        f = 4 if case["fp32"] else 8
        return {"bytes": 1300 * NEWTON * c * (f * m * m + 8 * m * 8 + 24 * m),
                "flops": 3 * c * _bdf_flops(m, 1.5 * m)}
    if kind == "imex":
        # 33 steps of 4 stages, one preconditioned Krylov iteration per Newton
        # iteration: state, stage vectors, J v and the 3 x 3 solve
        return {"bytes": 33 * 6 * 3 * case["n"] ** 3 * 8 * 12, "flops": 33 * 6 * case["n"] ** 3 * 150}
    macs = 144 * 128 + 128 * 128 + 128 * 64
    return {"bytes": case["steps"] * (case["batch"] * 4 * (144 + 64 + 64) + 28 * NPARAM),
            "flops": case["steps"] * 6.0 * macs * case["batch"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("vector", "krylov", "chem"):
        # sums in 64 bits in another order
        return {"rel": 1e-12, "max": 1e-9}
    if kind == "lu":
        # the Newton matrices' condition times the factors' rounding
        return {"rel": 1e-5, "max": 1e-2} if case["fp32"] else {"rel": 1e-12, "max": 1e-9}
    if kind in ("bucket", "batch"):
        # double precision follows the reference integrator bit for bit; with
        # single-precision factors the step sequences differ, and the states by
        # the integration's own error at rtol 1e-6
        return {"rel": 5e-6, "max": 2e-4} if case["fp32"] else "exact"
    if kind == "coupled":
        # sums in another order lead to another step sequence
        return {"rel": 1e-6, "max": 1e-4}
    if kind == "imex":
        # the same steps and iterations: sums in another order, or another
        # rounding of the single-precision preconditioner
        return {"rel": 2e-11, "max": 2e-9} if case["fp32"] else {"rel": 1e-12, "max": 1e-10}
    # bf16 products; Adam's first steps divide a gradient by its own size
    return {"rel": 2e-3, "max": 0.3}
