"""Eigen-solver and bond split without a warm start, across the sizes at which
the QR iteration in front of the Jacobi sweeps starts (33), changes its panel
(order 96, rows 32, 256, 512, 1024), takes first-order steps (129) or ends (complex above 1536).

Tolerances: the off-diagonal criterion and N eps |H| of rounding leave
eigenvalues to 1e-12 |H| and residuals to 1e-11 sqrt(N) |H| (the bounds of the
smaller sizes); each QR step and sweep loses a few eps of orthogonality per
vector, 1e-12 sqrt(N) in the Frobenius norm.
"""
import numpy as np
import pytest

from conftest import rand, rel_err

pytestmark = pytest.mark.gpu


def _spectrum(kind, N, rng):
    if kind == "graded":       # a density matrix: squared Schmidt values
        return np.logspace(0, -14, N)
    if kind == "degenerate":   # multiplets, and an exact null space
        lam = np.repeat(rng.uniform(0.1, 1.0, N // 8 + 1), 8)[:N]
        lam[N // 2:] = 0.0
        return lam
    return rng.uniform(-3, 3, N)


SIZES = ([(n, c, k) for n in (32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 257, 511, 545) for c in (False, True)
          for k in ("graded", "degenerate", "indefinite")]
         + [(1057, False, "graded"), (1057, False, "degenerate"), (1100, True, "graded"),
            (1536, True, "degenerate"), (1537, True, "graded"), (2048, False, "graded")])


@pytest.mark.parametrize("N,cplx,kind", SIZES)
def test_heig(dmrg_amd, ops, N, cplx, kind):
    rng = np.random.default_rng(N + (7 if cplx else 0))
    Q = np.linalg.qr(rand(rng, (N, N), cplx))[0]
    lam = _spectrum(kind, N, rng)
    H = (Q * lam) @ Q.conj().T
    H = (H + H.conj().T) / 2
    ev, vec, _ = ops.heig(dmrg_amd.DeviceArray.from_numpy(H))
    scale = np.abs(lam).max()
    assert np.max(np.abs(ev - np.sort(lam)[::-1])) < 1e-12 * scale
    assert np.linalg.norm(vec.conj().T @ vec - np.eye(N)) < 1e-12 * np.sqrt(N)
    assert np.linalg.norm(H @ vec - vec * ev) < 1e-11 * scale * np.sqrt(N)


@pytest.mark.parametrize("shape", ["diagonal", "block", "columns"])
def test_structured(dmrg_amd, ops, shape):
    """Zero columns below the diagonal (no reflection), zero-padded blocks and a
    rank-one matrix: eigenvalues by construction, orthonormal vectors."""
    N = 200
    rng = np.random.default_rng(3)
    if shape == "diagonal":
        H = np.diag(rng.uniform(-1, 1, N))
    elif shape == "block":
        H = np.zeros((N, N))
        B = rand(rng, (60, 60), False)
        H[100:160, 100:160] = B + B.T
    else:
        v = rand(rng, (N, 1), False)
        H = v @ v.T
    ev, vec, _ = ops.heig(dmrg_amd.DeviceArray.from_numpy(H))
    scale = np.linalg.norm(H, 2)
    assert np.max(np.abs(ev - np.sort(np.linalg.eigvalsh(H))[::-1])) < 1e-12 * scale
    assert np.linalg.norm(vec.T @ vec - np.eye(N)) < 1e-12 * np.sqrt(N)
    assert np.linalg.norm(H @ vec - vec * ev) < 1e-11 * scale * np.sqrt(N)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("scale_left", [False, True])
@pytest.mark.parametrize("m,n,k", [(129, 400, 100), (300, 161, 80), (520, 530, 256)])
def test_split_truncated(dmrg_amd, ops, cplx, scale_left, m, n, k):
    """Truncated split of a graded matrix: kept singular values to 1e-10 of
    themselves (a Gram matrix resolves eps sigma_1^2 / sigma_k^2, sigma_k >= 1e-2.5),
    and the discarded weight that of LAPACK's."""
    rng = np.random.default_rng(m + n + 2 * cplx + scale_left)
    r = min(m, n)
    s = np.logspace(0, -5, r)
    U = np.linalg.qr(rand(rng, (m, r), cplx))[0]
    V = np.linalg.qr(rand(rng, (n, r), cplx))[0]
    M = (U * s) @ V.conj().T
    k = min(k, r // 2)
    left, right, sig, nk = ops.svd_split(dmrg_amd.DeviceArray.from_numpy(M), k, scale_left=scale_left)
    assert nk == k
    assert np.max(np.abs(sig[:k] - s[:k]) / s[:k]) < 1e-10
    iso = right.conj().T if scale_left else left
    assert np.linalg.norm(iso.conj().T @ iso - np.eye(k)) < 1e-12 * np.sqrt(k) * 10
    err = np.linalg.norm(M - left @ right)
    assert abs(err - np.linalg.norm(s[k:])) < 1e-10
    assert rel_err(left @ right, (U[:, :k] * s[:k]) @ V[:, :k].conj().T) < 1e-8
