"""The 64x32 and 64x64 tiles of the GEMM at ragged sizes, odd offsets and leading
dimensions, inside NaN (545 x 547 takes 64x32 tiles in the real types, 1407 x 1405
64x64 ones in all), with and without adding to C: these tiles read and write two
rows of an operand that is contiguous along m at a time.  Tolerances as for the
small tiles (at most 35 terms here).
"""
import numpy as np
import pytest

from test_gpu_gemm_tiles import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(545, 547), (546, 544), (1407, 1405), (1408, 1409)])
@pytest.mark.parametrize("K,off,pad,beta", [(1, 1, 1, 0.5), (19, 0, 0, 0.0), (34, 3, 2, 0.5)])
def test_real(dmrg_amd, ops, M, N, K, off, pad, beta):
    for opA, opB in ((0, 0), (1, 0), (0, 1), (1, 1)):
        assert _run(dmrg_amd, ops, np.float64, opA, opB, M, N, K, off, pad, beta) < 1e-13, (opA, opB)
        assert _run(dmrg_amd, ops, np.float32, opA, opB, M, N, K, off, pad, 0.0) < 1e-5, (opA, opB)


@pytest.mark.parametrize("opA,opB", [(0, 0), (3, 0), (0, 3), (2, 1)])
@pytest.mark.parametrize("K,off,pad,beta", [(1, 1, 1, 0.5), (19, 0, 0, 0.0)])
def test_complex(dmrg_amd, ops, opA, opB, K, off, pad, beta):
    assert _run(dmrg_amd, ops, np.complex128, opA, opB, 1407, 1405, K, off, pad, beta) < 1e-13
