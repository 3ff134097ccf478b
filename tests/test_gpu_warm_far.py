"""Warm splits that start far from their basis (the second sweep of a run) or
whose block overlap has no polar factor, at block sizes on either side of the
limits of the QR iteration (order 64 of the padded block) and of its panels.

The run with warm starts must end in the state of the run without: energies of
the last sweep to 1e-8 of themselves (both are at the fixed point of the
truncated sweep, whose energy is stationary: the truncated weight is below 1e-8
here) and a state of unit norm to 1e-10.
"""
import numpy as np
import pytest

from oracle import models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx,chi", [(False, 12), (False, 33), (False, 48), (False, 64), (False, 100), (True, 16),
                                      (True, 30)])
def test_warm_ends_like_cold(dmrg_amd, cplx, chi):
    L = 14 if not cplx else 8
    Ws = models.heisenberg_mpo(L) if not cplx else models.josephson_mpo(L, n_max=1)
    D, d = Ws[0].shape[0], Ws[0].shape[1]
    E, norm = {}, {}
    for warm in (0, 1):
        eng = dmrg_amd.DMRG(L, d, chi, D, dtype="c128" if cplx else "f64", tol=0.0, krylov_max=30, svd_warm=warm)
        eng.set_mpo(Ws)
        eng.initialize_mps_random(seed=5, scale=0.1)
        eng.run(7)
        E[warm] = np.array(eng.sweep_energies())
        norm[warm] = eng.expectation()[1]
        st = eng.stats()
        assert (st["svd_warm_starts"] > 0) == bool(warm)
        eng.close()
    assert abs(E[1][-1] - E[0][-1]) < 1e-8 * abs(E[0][-1])
    assert all(abs(n - 1) < 1e-10 for n in norm.values())


@pytest.mark.parametrize("seed", [31, 34])
def test_full_rank_bonds_keep_their_size(dmrg_amd, seed):
    """Bonds that are not truncated keep every vector: their smallest Schmidt
    values are of rounding size, and a warm split must not resolve them below
    the cutoff where the sweeps leave them mixed with the rest."""
    L, chi = 32, 256
    Ws = models.heisenberg_mpo(L)
    with dmrg_amd.DMRG(L, 2, chi, 5, tol=0.0, krylov_max=20) as eng:
        eng.set_mpo(Ws)
        eng.initialize_mps_random(seed=seed, scale=0.1)
        eng.run(4)
        assert list(eng.bond_dims()) == [min(2 ** i, 2 ** (L - i), chi) for i in range(L + 1)]
