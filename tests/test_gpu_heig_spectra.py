"""Eigen-solves on either side of the limits that choose their path: order 96 and
97 (QR steps from a padded order of 128), 128 and 129 (first-order steps from
160), the part of the spectrum that carries a positive semidefinite matrix (1/25
to 3/5 of it: QR steps), and spectra with many zeros (two inner sweeps a block pair).

The iteration stops once every coupling is below 1e-14 |H|_F, so an eigenvalue is
within (N - 1) 1e-14 |H|_F of its row sum's centre, plus the rounding of some 20
sweeps of N unitary updates, at most about 20 N eps: 5e-12 |H|_F covers both at
N = 330, and 5e-12 the orthogonality of the vectors.
"""
import numpy as np
import pytest

from conftest import rand

pytestmark = pytest.mark.gpu
TOL = 5e-12


def spectrum(kind, n):
    zeros = lambda r: np.zeros(n - r)
    return {
        "graded": lambda: np.logspace(0, -9, n),
        "part-below": lambda: np.r_[np.ones(max(1, n // 27)), zeros(max(1, n // 27))],
        "part-above-low": lambda: np.r_[np.ones(n // 20), zeros(n // 20)],
        "part-below-high": lambda: np.r_[np.ones(n // 2), zeros(n // 2)],
        "part-above-high": lambda: np.r_[np.ones(2 * n // 3), zeros(2 * n // 3)],
        "signs": lambda: np.r_[np.ones(n // 8), -np.ones(n // 8), zeros(2 * (n // 8))],
        "negative": lambda: -np.logspace(0, -9, n),
        "one": lambda: np.r_[1.0, zeros(1)],
    }[kind]()


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("kind", ["graded", "part-below", "part-above-low", "part-below-high", "part-above-high",
                                  "signs", "negative", "one"])
@pytest.mark.parametrize("n", [96, 97, 128, 129, 160, 161, 330])
def test_heig_spectra(dmrg_amd, ops, n, kind, cplx):
    rng = np.random.default_rng(n)
    U = np.linalg.qr(rand(rng, (n, n), cplx))[0]
    s = np.sort(spectrum(kind, n))[::-1]
    H = (U * s) @ U.conj().T
    H = (H + H.conj().T) / 2
    ev, V, _ = ops.heig(dmrg_amd.DeviceArray.from_numpy(H))
    fro = np.linalg.norm(H)
    assert np.max(np.abs(ev - s)) < TOL * fro
    assert np.max(np.abs(V.conj().T @ V - np.eye(n))) < TOL
    assert np.linalg.norm(H @ V - V * ev) < TOL * fro * np.sqrt(n)
