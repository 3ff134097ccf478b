"""The split-BF16 product at the edges of its tiles (64 x 64, 32 values of k),
with odd leading dimensions and addresses inside arrays of NaN, and the matvec
whose products are cut along k.

Tolerance: the three bf16 terms carry 24 bits and the six products leave 2^-24
of |a||b|, so with FP32 sums of up to 300 terms of order one the error is that of
an FP32 product: 1e-5 in norm for the product (as for FP32), 2e-5 for the two
products and the MPO step of the matvec.
"""
import numpy as np
import pytest

from conftest import rand, rel_err
from oracle import dmrg as od
from test_gpu_gemm_tiles import _embed

pytestmark = pytest.mark.gpu

EDGES = [(1, 1, 1), (3, 2, 31), (64, 64, 32), (65, 63, 33), (63, 65, 63), (16, 130, 64), (129, 17, 65), (70, 66, 95),
         (2, 3, 96), (64, 1, 97), (33, 100, 127), (100, 33, 128), (65, 65, 160), (40, 90, 300)]


@pytest.mark.parametrize("M,N,K", EDGES)
def test_edges(dmrg_amd, ops, M, N, K):
    lib = dmrg_amd.lib()
    rng = np.random.default_rng(M + 100 * N + 10000 * K)
    for off, pad in ((0, 0), (1, 1), (3, 2)):
        for opA, opB in ((0, 0), (1, 0), (0, 1), (1, 1)):
            A = rand(rng, (K, M) if opA else (M, K), False).astype(np.float32)
            B = rand(rng, (N, K) if opB else (K, N), False).astype(np.float32)
            C = np.zeros((M, N), np.float32)
            pa, lda, ka = _embed(dmrg_amd, A, np.float32, off, pad)
            pb, ldb, kb = _embed(dmrg_amd, B, np.float32, off + 1, pad + 2)
            pc, ldc, kc = _embed(dmrg_amd, C, np.float32, off, pad)
            rc = lib.dmrg_op_gemm_f32(ops._h, None, dmrg_amd.PREC_BF16X3, opA, opB, M, N, K, pa, lda, pb, ldb, pc, ldc)
            assert rc == dmrg_amd.OK, lib.dmrg_last_error()
            out = kc.numpy()
            got = np.stack([out[off + j * ldc: off + j * ldc + M] for j in range(N)], axis=1)
            ref = (A.T if opA else A).astype(float) @ (B.T if opB else B).astype(float)
            assert rel_err(got.astype(float), ref) < 1e-5, (off, opA, opB)
            out[np.concatenate([np.arange(off + j * ldc, off + j * ldc + M) for j in range(N)])] = np.nan
            assert np.isnan(out).all()  # nothing written outside C


@pytest.mark.parametrize("cL,cR,D", [(1, 300, 5), (30, 200, 5), (33, 65, 11), (40, 129, 7), (301, 77, 5)])
def test_sliced_matvec(dmrg_amd, ops, cL, cR, D):
    rng = np.random.default_rng(cL + cR + D)
    f32 = lambda x: x.astype(np.float32)  # noqa: E731
    L, R, th = (f32(rand(rng, s, False)) for s in ((cL, D, cL), (cR, D, cR), (cL, 2, 2, cR)))
    W = rand(rng, (D, 2, 2, D), False)
    dev = dmrg_amd.DeviceArray.from_numpy
    out = dmrg_amd.DeviceArray(th.shape, np.float32)
    ops.heff2_f32(dev(L, np.float32), dev(R, np.float32), dev(W), dev(W), dev(th, np.float32), out,
                  prec=dmrg_amd.PREC_BF16X3)
    ref = od.apply_heff2(L.astype(float), R.astype(float), W, W, th.astype(float))
    assert rel_err(out.numpy().astype(float), ref) < 2e-5
