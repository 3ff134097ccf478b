"""Eigen-solver and bond split of matrices whose norm is far from one.

An eigenvalue problem times a power of two is the same problem: the results
must be those of the unscaled one, to the tolerances of the cold splits
(eigenvalues 1e-12 |H|, residuals 1e-11 sqrt(N) |H|, orthonormality 1e-12
sqrt(N)); 2^-465 is 1e-140, 2^-485 1e-146, where squares of rounding-size
entries leave the range of a double.
"""
import numpy as np
import pytest

from conftest import rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [-485, -465, 465])
@pytest.mark.parametrize("kind", ["graded", "flat"])
@pytest.mark.parametrize("N,cplx", [(n, c) for n in (33, 64, 200, 512) for c in (False, True)])
def test_heig_scaled(dmrg_amd, ops, N, cplx, kind, p):
    rng = np.random.default_rng(N + cplx)
    Q = np.linalg.qr(rand(rng, (N, N), cplx))[0]
    lam = np.logspace(0, -14, N) if kind == "graded" else rng.uniform(0.1, 1.0, N)
    H = (Q * lam) @ Q.conj().T
    H = (H + H.conj().T) / 2
    ev, vec, _ = ops.heig(dmrg_amd.DeviceArray.from_numpy(H * 2.0 ** p))
    ev = ev * 2.0 ** -p
    assert np.max(np.abs(ev - np.sort(lam)[::-1])) < 1e-12
    assert np.linalg.norm(vec.conj().T @ vec - np.eye(N)) < 1e-12 * np.sqrt(N)
    assert np.linalg.norm(H @ vec - vec * ev) < 1e-11 * np.sqrt(N)


@pytest.mark.parametrize("p", [-242, -232, 232])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("left", [False, True])
def test_split_scaled(dmrg_amd, ops, cplx, left, p):
    """Kept singular values to 1e-10 of themselves (sigma_k >= 1e-2.5 of the
    largest), the product to that of LAPACK's truncation."""
    m, n, k = 129, 160, 60
    rng = np.random.default_rng(7 + cplx)
    U = np.linalg.qr(rand(rng, (m, m), cplx))[0]
    V = np.linalg.qr(rand(rng, (n, m), cplx))[0]
    s = np.logspace(0, -5, m)
    M = (U * s) @ V.conj().T
    lt, rt, sig, nk = ops.svd_split(dmrg_amd.DeviceArray.from_numpy(M * 2.0 ** p), k, cutoff=0.0, scale_left=left)
    assert nk == k
    assert np.max(np.abs(sig * 2.0 ** -p - s[:k]) / s[:k]) < 1e-10
    iso = rt.conj().T if left else lt
    assert np.linalg.norm(iso.conj().T @ iso - np.eye(k)) < 1e-12 * np.sqrt(k) * 10
    assert np.linalg.norm((lt @ rt) * 2.0 ** -p - (U[:, :k] * s[:k]) @ V[:, :k].conj().T) < 1e-8
