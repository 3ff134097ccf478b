"""The rank of splits without a warm start: bonds that are not truncated keep
every vector, as they do with the sweeps alone, and the rank of a matrix whose
Schmidt values end in a gap is the number above it.
"""
import numpy as np
import pytest

from conftest import rand
from oracle import models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 2])
def test_full_rank_bonds_keep_their_size(dmrg_amd, seed):
    L, chi = 32, 256
    with dmrg_amd.DMRG(L, 2, chi, 5, tol=0.0, krylov_max=20, svd_warm=0) as eng:
        eng.set_mpo(models.heisenberg_mpo(L))
        eng.initialize_mps_random(seed=seed, scale=0.1)
        eng.run(3)
        assert eng.stats()["svd_warm_starts"] == 0
        assert list(eng.bond_dims()) == [min(2 ** i, 2 ** (L - i), chi) for i in range(L + 1)]


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_single_site_bonds_with_a_cutoff(dmrg_amd, seed):
    """Single-site splits start cold every time and cannot grow a bond again."""
    L, chi = 16, 64
    with dmrg_amd.DMRG(L, 2, chi, 5, tol=0.0, krylov_max=20, variant=dmrg_amd.SINGLE_SITE, svd_cutoff=1e-10) as eng:
        eng.set_mpo(models.heisenberg_mpo(L))
        eng.initialize_mps_random(seed=seed, scale=0.1)
        eng.run(2)
        assert list(eng.bond_dims()) == [min(2 ** i, 2 ** (L - i), chi) for i in range(L + 1)]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("left", [False, True])
@pytest.mark.parametrize("m,n,r", [(40, 50, 7), (130, 100, 30), (300, 260, 64)])
def test_rank_ends_in_a_gap(dmrg_amd, ops, cplx, left, m, n, r):
    """Product of two factors of r vectors: exactly r singular values above
    rounding (sigma_r >= 1e-2 sigma_1 by construction, the rest <= 1e-15)."""
    rng = np.random.default_rng(m + r + cplx)
    U = np.linalg.qr(rand(rng, (m, r), cplx))[0]
    V = np.linalg.qr(rand(rng, (n, r), cplx))[0]
    s = np.logspace(0, -2, r)
    M = (U * s) @ V.conj().T
    _, _, sig, nk = ops.svd_split(dmrg_amd.DeviceArray.from_numpy(M), min(m, n) // 2, cutoff=1e-13, scale_left=left)
    assert nk == r
    assert np.max(np.abs(sig - s) / s) < 1e-10
