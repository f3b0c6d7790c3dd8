"""Mass-action right-hand side and Jacobian kernels where their reactions and
terms leave the fast part: more than two reactions per lane (R > 2 pow2ceil(m),
whose further rates are read where they are used), more than twelve terms per
species (the rest are read from LDS), one species, several cells per group with
a partial last round, and a Jacobian array on an odd 8-byte place (single
stores in place of pairs).  Bit for bit the serial evaluation; a state that is
not finite stays in its cell."""
import ctypes as C

import numpy as np
import pytest

from sundials_amd import _lib
from helpers import dp

pytestmark = pytest.mark.gpu

# (m, R), few cells, and more cells than the widest launch has groups
CASES = [(1, 5, 130, 2100007), (3, 20, 37, 530003), (5, 40, 19, 270001), (16, 80, 7, 120001),
         (64, 160, 3, 5003)]


def _eval(m, R, ncells, odd_place):
    import torch

    core, hip = _lib.core(), _lib.hip()
    base = core.SUNAMD_MassActionCreate(m, R, min(ncells, 499), 40 + m, 0.2)
    p = core.SUNAMD_MassActionTile(base, ncells)
    core.SUNAMD_MassActionFree(base)
    y = np.ctypeslib.as_array(p.contents.y0, shape=(ncells * m,)).copy()
    y *= np.random.default_rng(m).uniform(0.5, 1.5, y.size)
    y[-1] = np.nan
    y[(ncells // 2) * m] = np.inf
    f_ref, J_ref = np.zeros(ncells * m), np.zeros(ncells * m * m)
    core.SUNAMD_MassActionRhsHost(p, dp(y), dp(f_ref), 0, ncells)
    core.SUNAMD_MassActionJacHost(p, dp(y), dp(J_ref), 0, ncells)
    terms = np.bincount(np.ctypeslib.as_array(p.contents.idx, shape=(4 * R,)), minlength=m)
    dev = hip.SUNAMD_MassActionToDevice(p, C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert dev
    ty = torch.from_numpy(y).cuda()
    tf = torch.full((y.size,), 7.0, dtype=torch.float64, device="cuda")
    tJ = torch.full((J_ref.size + 2,), 7.0, dtype=torch.float64, device="cuda")
    at = 1 if odd_place else 0
    assert hip.SUNAMD_MassActionRhsDevArrays(dev, C.c_void_p(ty.data_ptr()),
                                             C.c_void_p(tf.data_ptr())) == 0
    assert hip.SUNAMD_MassActionJacDevArrays(dev, C.c_void_p(ty.data_ptr()),
                                             C.c_void_p(tJ.data_ptr() + 8 * at)) == 0
    torch.cuda.synchronize()
    f, J = tf.cpu().numpy(), tJ.cpu().numpy()
    hip.SUNAMD_MassActionDevFree(dev)
    core.SUNAMD_MassActionFree(p)
    # nothing written beside the Jacobian
    assert (J[:at] == 7.0).all() and (J[at + J_ref.size:] == 7.0).all()
    return terms, (f, f_ref), (J[at:at + J_ref.size], J_ref)


@pytest.mark.parametrize("odd_place", [False, True])
@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("m,R,few,lots", CASES)
def test_many_reactions_per_species(m, R, few, lots, many, odd_place):
    terms, f, J = _eval(m, R, lots if many else few, odd_place)
    group = 1 << (m - 1).bit_length()
    assert R > 2 * group and terms.max() > 12
    for got, ref in (f, J):
        assert np.array_equal(got, ref, equal_nan=True)
