"""Splits and eigen-solves of what is diagonal already: no sweep is needed.

Diagonal, isometric (equal Schmidt values: rho is the identity) and block
matrices, whose kept group by diagonal entries is not the dominant one: only a
matrix without couplings at all may be taken as it came.
"""
import numpy as np
import pytest

from conftest import rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("N", [33, 64, 100, 257])
def test_diagonal_takes_no_sweep(dmrg_amd, ops, cplx, N):
    rng = np.random.default_rng(N)
    lam = rng.uniform(-1, 1, N)
    ev, vec, sweeps = ops.heig(dmrg_amd.DeviceArray.from_numpy(np.diag(lam).astype(complex if cplx else float)))
    assert sweeps == 0
    assert np.array_equal(ev, np.sort(lam)[::-1])
    assert np.array_equal(np.abs(vec), np.eye(N)[:, np.argsort(-lam, kind="stable")])


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("m,n,k", [(40, 50, 20), (100, 100, 100), (200, 300, 77)])
def test_isometry(dmrg_amd, ops, cplx, m, n, k):
    """Singular values all one, to N eps of the product that forms rho."""
    rng = np.random.default_rng(m + k)
    M = np.linalg.qr(rand(rng, (n, m), cplx))[0].conj().T
    left, right, sig, nk = ops.svd_split(dmrg_amd.DeviceArray.from_numpy(np.ascontiguousarray(M)), k)
    assert nk == k
    assert np.max(np.abs(sig - 1)) < 1e-13
    assert np.linalg.norm(left.conj().T @ left - np.eye(k)) < 1e-12 * np.sqrt(k)
    assert np.linalg.norm(left @ right - left @ (left.conj().T @ M)) < 1e-12 * np.sqrt(k)


@pytest.mark.parametrize("left", [False, True])
def test_block_below_the_cut_is_found(dmrg_amd, ops, left):
    """rho = diag(0.5, 0.3, ...) + a block of 40 entries 0.02: by diagonal entries
    the kept group decouples from the block, whose eigenvalue 0.8 leads."""
    N, k = 64, 8
    G = np.diag(np.concatenate([np.linspace(0.5, 0.3, 24), np.zeros(40)]))
    G[24:, 24:] = 0.02
    w, v = np.linalg.eigh(G)
    M = (v * np.sqrt(np.clip(w, 0, None))) @ v.T
    lt, rt, sig, nk = ops.svd_split(dmrg_amd.DeviceArray.from_numpy(M), k, scale_left=left)
    assert nk == k
    assert abs(np.linalg.norm(lt @ rt) ** 2 - np.sort(w)[::-1][:k].sum()) < 1e-12
