"""Products of more columns than one launch has workgroups for (65535 tiles of
32).  Integers, so that every sum is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 65535 * 32


@pytest.mark.parametrize("M,K", [(1, 1), (2, 3), (33, 2)])
@pytest.mark.parametrize("n", [N, N + 1, N + 31000])
@pytest.mark.parametrize("cplx,opB", [(False, 0), (False, 1), (True, 3)])
def test_many_columns(dmrg_amd, ops, M, K, n, cplx, opB):
    rng = np.random.default_rng(M + K)
    ints = lambda s: rng.integers(-8, 9, s) + (1j * rng.integers(-8, 9, s) if cplx else 0.0)
    A, B = ints((M, K)), ints((n, K) if opB else (K, n))
    C = dmrg_amd.DeviceArray((M, n), A.dtype)
    ops.gemm(0, opB, dmrg_amd.DeviceArray.from_numpy(A), dmrg_amd.DeviceArray.from_numpy(B), C)
    ref = A @ (B.conj().T if opB == 3 else B.T if opB else B)
    assert np.array_equal(C.numpy(), ref)
