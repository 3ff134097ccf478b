"""Lanczos vectors of more than 512 workgroups (2^21 elements), whose sums over
the workgroups are formed by launches of their own.

As for the shorter lengths: energy against the oracle's Lanczos of as many steps
and against the Rayleigh quotient to 1e-11 |H|, unit norm to 1e-13.  A start of
zero norm is the seeded stream in both.
"""
import numpy as np
import pytest

from conftest import rand
from oracle import dmrg as od

pytestmark = pytest.mark.gpu


def _herm(rng, c, cplx):
    x = rand(rng, (c, 1, c), cplx)
    return (x + np.conj(np.swapaxes(x, 0, 2))) / (2 * np.sqrt(c))


@pytest.mark.parametrize("cL,cR,cplx,zero", [(724, 724, False, False), (725, 724, False, False), (725, 724, False, True),
                                             (725, 724, True, False), (1100, 1000, False, False)])
def test_lanczos_long(dmrg_amd, ops, cL, cR, cplx, zero):
    rng = np.random.default_rng(cL + cplx)
    L, R = _herm(rng, cL, cplx), _herm(rng, cR, cplx)
    W = np.zeros((1, 2, 2, 1), L.dtype)
    W[0, :, :, 0] = [[1.0, 0.3], [0.3, -0.5]]
    th = np.zeros((cL, 2, 2, cR), L.dtype) if zero else rand(rng, (cL, 2, 2, cR), cplx)
    H = lambda x: od.apply_heff2(L, R, W, W, x)
    dev = dmrg_amd.DeviceArray.from_numpy
    dth = dev(th)
    E, nit = ops.lanczos2(dev(L), dev(R), dev(W), dev(W), dth, krylov_max=5, site=2)
    psi = dth.numpy()
    Hpsi = H(psi)
    E_ref, _ = od.lanczos(H, th, 2, 5)
    scale = max(np.linalg.norm(Hpsi), 1.0)
    assert nit == 5
    assert abs(np.linalg.norm(psi) - 1) < 1e-13
    assert abs(np.vdot(psi, Hpsi).real - E) < 1e-11 * scale
    assert abs(E - E_ref) < 1e-11 * scale
