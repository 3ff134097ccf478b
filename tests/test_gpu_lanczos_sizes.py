"""The Lanczos vector kernels where their launch changes: one workgroup up to
2048 elements (1 or 2 a thread), then 1, 2 or 4 elements a thread from 2^18 and
2^19 on, and more than 256 workgroups past 2^20.

H_eff is built Hermitian from Hermitian factors.  The energy is compared with
the oracle's Lanczos of as many steps from the same start: with one full
projection each keeps its basis orthogonal to a few eps, so the Ritz values
agree to k eps |H| (bound 1e-11 |H|); the returned vector has unit norm to
1e-13 and the Rayleigh quotient E to the same 1e-11 |H|.
"""
import numpy as np
import pytest

from conftest import rand
from oracle import dmrg as od

pytestmark = pytest.mark.gpu


def _herm(rng, shape, ax, cplx):
    x = rand(rng, shape, cplx)
    return (x + np.conj(np.swapaxes(x, *ax))) / 2


# cL, cR, d, Krylov steps; n = cL d^2 cR
SIZES = [(1, 1, 1, 4), (3, 1, 1, 5), (3, 7, 1, 12), (33, 31, 1, 40), (16, 16, 2, 9), (41, 25, 1, 17), (31, 33, 1, 17),
         (16, 32, 2, 33), (27, 19, 2, 16), (49, 41, 1, 8), (63, 65, 1, 24), (70, 59, 1, 10)]
LARGE = [(256, 256, 2, 9), (257, 256, 2, 9), (362, 362, 2, 10), (363, 363, 2, 7), (512, 512, 2, 9), (513, 512, 2, 9)]


@pytest.mark.parametrize("cL,cR,d,kmax,cplx", [s + (c,) for s in SIZES for c in (False, True)]
                         + [s + (False,) for s in LARGE] + [(257, 256, 2, 7, True), (363, 363, 2, 5, True)])
def test_lanczos_lengths(dmrg_amd, ops, cL, cR, d, kmax, cplx):
    rng = np.random.default_rng(cL * 1000 + cR * 10 + cplx)
    D = 2
    L = _herm(rng, (cL, D, cL), (0, 2), cplx) / np.sqrt(cL)
    R = _herm(rng, (cR, D, cR), (0, 2), cplx) / np.sqrt(cR)
    W1 = _herm(rng, (D, d, d, D), (1, 2), cplx)
    W2 = _herm(rng, (D, d, d, D), (1, 2), cplx)
    th = rand(rng, (cL, d, d, cR), cplx)
    H = lambda x: od.apply_heff2(L, R, W1, W2, x)
    dev = dmrg_amd.DeviceArray.from_numpy
    dth = dev(th)
    E, nit = ops.lanczos2(dev(L), dev(R), dev(W1), dev(W2), dth, krylov_max=kmax, site=2)
    psi = dth.numpy()
    Hpsi = H(psi)
    scale = max(np.linalg.norm(Hpsi), np.linalg.norm(H(th)) / np.linalg.norm(th))
    E_ref, _ = od.lanczos(H, th, 2, kmax)
    assert 1 <= nit <= kmax
    assert abs(np.linalg.norm(psi) - 1) < 1e-13
    assert abs(np.vdot(psi, Hpsi).real - E) < 1e-11 * scale
    assert abs(E - E_ref) < 1e-11 * scale


def _lowest(a, b):
    """Lowest eigenvalue by bisection on the pivots of T - x in extended
    precision (LAPACK's tridiagonal solvers are off by up to 9e-15 here)."""
    a, b2 = a.astype(np.longdouble), b.astype(np.longdouble) ** 2
    lo, hi = a.min() - 2 * np.sqrt(b2.max()), a.min()
    for _ in range(80):
        x = (lo + hi) / 2
        q = a[0] - x
        for i in range(1, len(a)):
            if q <= 0:
                break
            q = (a[i] - x) - b2[i - 1] / q
        lo, hi = (lo, x) if q <= 0 else (x, hi)
    return lo


@pytest.mark.parametrize("k", [2, 7, 8, 9, 16, 17, 63, 64, 65, 127, 128])
@pytest.mark.parametrize("kind", ["plain", "huge", "small", "split", "graded", "shifted"])
def test_tridiagonal(ops, k, kind):
    """Lowest eigenvalue of a tridiagonal to 4 eps |T| (bisection ends at 2 eps;
    one more of rounding either side), residual of its vector to 1e-13 |T|."""
    rng = np.random.default_rng(k)
    a = rng.uniform(-2, 2, k)
    b = rng.uniform(0.1, 1.0, k - 1)
    if kind == "huge":
        a, b = a * 1e150, b * 1e150
    elif kind == "small":
        a, b = a * 1e-150, b * 1e-150
    elif kind == "split":
        b[::3] = 0.0
    elif kind == "graded":
        b *= np.logspace(0, -14, k - 1)
    elif kind == "shifted":
        a += 1e6
    lam, y = ops.tridiag_lowest(a, b)
    s = max(np.abs(a).max(), np.abs(b).max())
    norm = 3.0
    assert abs(lam / s - _lowest(a / s, b / s)) < 4 * np.finfo(float).eps * norm
    T = np.diag(a / s) + np.diag(b / s, 1) + np.diag(b / s, -1)
    assert abs(np.linalg.norm(y) - 1) < 1e-13
    assert np.linalg.norm(T @ y - (lam / s) * y) < 1e-13 * norm
