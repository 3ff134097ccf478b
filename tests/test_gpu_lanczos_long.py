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
from oracle.prng import uniform_pm1

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


def test_lanczos_past_32_bit_indices(dmrg_amd):
    """2^32 + 2^20 elements (160 GiB of vectors): H_eff is the identity and the
    start has zero norm, so the result is the seeded stream over its norm, with
    energy one.  Each element to 1e-14 of one factor, which is 1/sqrt(n/3) to the
    1e-4 that n samples of a variance leave many times over."""
    cL, cR, d = 4096, 4097, 16
    n = cL * d * d * cR
    dev, L = dmrg_amd.DeviceArray, dmrg_amd.lib()
    eye = lambda c: dev.from_numpy(np.eye(c).reshape(c, 1, c))
    W = dev.from_numpy(np.eye(d).reshape(1, d, d, 1))
    ops = dmrg_amd.Ops(0)
    try:
        theta = dev((cL, d, d, cR), np.float64)
        rest = [dev((cL, d, d, cR), np.float64) for _ in range(4)]  # room for the work vectors
        for x in rest:
            x.free()
    except dmrg_amd.DMRGError:
        pytest.skip("less than 180 GB of device memory free")
    at = lambda i: theta.ptr.value + 8 * i
    zeros = np.zeros(2 ** 20)
    dmrg_amd._check(L.dmrg_memcpy_h2d(at(0), zeros.ctypes.data, zeros.nbytes))
    done = zeros.size
    while done < n:
        k = min(done, n - done)
        dmrg_amd._check(L.dmrg_memcpy_d2d(at(done), at(0), 8 * k))
        done += k
    E, nit = ops.lanczos2(eye(cL), eye(cR), W, W, theta, krylov_max=1, site=3)
    f = []
    for i in (0, 2 ** 20, 2 ** 31 - 500, 2 ** 32 - 500, 2 ** 32 + 12345, n - 1000):
        got = np.empty(1000)
        dmrg_amd._check(L.dmrg_memcpy_d2h(got.ctypes.data, at(i), got.nbytes))
        ref = uniform_pm1(42 + 3, 1000, offset=i)
        f.append(got @ ref / (ref @ ref))
        assert np.max(np.abs(got - f[-1] * ref)) < 1e-14 * f[0]
    theta.free()
    ops.close()
    assert nit == 1 and abs(E - 1) < 1e-12
    assert np.ptp(f) < 1e-14 * f[0]
    assert abs(f[0] * np.sqrt(n / 3) - 1) < 1e-4
