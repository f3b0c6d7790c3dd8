"""The two-launch training step at the sizes where it can go wrong: one block
of 16 rows, an odd number of blocks (the last 32-deep slice of the weight
gradients half empty), more slices than a wavefront keeps in flight, and more
steps than one mask-sum launch covers.  Gradients against the float64 reference
that rounds to bf16 at the same points (differences: FP32 accumulation, and a
bf16 rounding it turns over, 2^-8 of one term of the sum); the update against
Adam in numpy float32 from the gradient the library returns."""
import ctypes as C

import numpy as np
import pytest

from mlp_ref import IN, IN_PAD, NPARAM, OUT, loss_grad, unpack
from sundials_amd import _lib

pytestmark = pytest.mark.gpu
PF = C.POINTER(C.c_float)


def _fp(a):
    return a.ctypes.data_as(PF)


def _data(n, seed):
    rng = np.random.default_rng(seed)
    x = np.zeros((n, IN_PAD), dtype=np.float32)
    x[:, :IN] = rng.uniform(-1.5, 0.5, (n, IN))
    t = rng.standard_normal((n, OUT)).astype(np.float32)
    mask = (rng.random((n, OUT)) < 0.6).astype(np.float32)
    return x, t, mask


def _grad(hip, M, x, t, mask):
    loss, g = C.c_float(), np.zeros(NPARAM, dtype=np.float32)
    assert hip.SUNAMD_MLPLossGrad(M, _fp(x), _fp(t), _fp(mask), len(x), C.byref(loss), _fp(g)) == 0
    return loss.value, g


def _train(hip, M, x, t, mask, batch, steps, lr=1e-3):
    import torch

    d = [torch.from_numpy(a).cuda() for a in (x, t, mask)]
    torch.cuda.synchronize()
    loss = C.c_float()
    assert hip.SUNAMD_MLPTrain(M, *(C.c_void_p(a.data_ptr()) for a in d), len(x), batch, steps, lr,
                               C.byref(loss)) == 0
    p = np.zeros(NPARAM, dtype=np.float32)
    assert hip.SUNAMD_MLPGetParams(M, _fp(p)) == 0
    return loss.value, p


@pytest.mark.parametrize("B", [16, 32, 48, 1024, 1040, 2064])
def test_gradient_and_update(B):
    hip = _lib.hip()
    M = hip.SUNAMD_MLPCreate(5, 2064)
    assert M
    try:
        # a larger batch first: what it leaves in the work arrays is not read
        _grad(hip, M, *_data(2064, 1))
        x, t, mask = _data(B, B)
        p0 = np.zeros(NPARAM, dtype=np.float32)
        assert hip.SUNAMD_MLPGetParams(M, _fp(p0)) == 0
        loss, g = _grad(hip, M, x, t, mask)
        l_ref, g_ref = loss_grad(p0.astype(np.float64), x, t, mask)
        assert abs(loss - l_ref) <= 1e-4 * abs(l_ref)
        gd, gr = unpack(g), unpack(g_ref)
        for name in gr:
            assert np.abs(gd[name] - gr[name]).max() <= 1e-2 * np.abs(gr[name]).max() + 1e-7, name
        l1, p1 = _train(hip, M, x, t, mask, B, 1)
        assert l1 == pytest.approx(loss, rel=1e-5)
        f = np.float32
        m, v = (f(1) - f(0.9)) * g, (f(1) - f(0.999)) * g * g
        step = f(1e-3) * (m / (f(1) - f(0.9))) / (np.sqrt(v / (f(1) - f(0.999))) + f(1e-8))
        # float32 rounding of the update's factors (1 - 0.999 alone: 3e-5)
        assert np.abs(p1 - (p0 - step)).max() <= 1e-3 * 1e-4 + 2.0 ** -23 * np.abs(p0).max()
    finally:
        hip.SUNAMD_MLPFree(M)


def test_steps_past_one_mask_sum_launch():
    hip = _lib.hip()
    x, t, mask = _data(48, 9)
    out = []
    for parts in ((300,), (130, 170)):
        M = hip.SUNAMD_MLPCreate(5, 48)
        assert M
        try:
            for s in parts:
                loss, p = _train(hip, M, x, t, mask, 48, s)
            out.append((loss, p))
        finally:
            hip.SUNAMD_MLPFree(M)
    # the same 300 steps on the same rows, bit for bit
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
