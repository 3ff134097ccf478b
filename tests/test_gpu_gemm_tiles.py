"""The GEMM kernels at the edges of their tiles and of their 16-byte chunks.

Operands sit inside larger arrays filled with NaN, at odd offsets and with odd
leading dimensions: a value read from outside an operand, or a chunk that
crosses the end of a row, shows as NaN or as an O(1) error.  Tolerances: FP64
1e-13 relative (at most 700 terms of order one, n eps = 1.6e-13 at worst,
sqrt(n) eps in the mean); FP32 1e-5 by the same count.
"""
import ctypes

import numpy as np
import pytest

from conftest import rand, rel_err
from oracle import dmrg as od

pytestmark = pytest.mark.gpu

EDGES = [(1, 1, 1), (1, 70, 2), (2, 3, 1), (3, 2, 5), (4, 4, 3), (15, 17, 16), (17, 15, 8), (31, 33, 7),
         (33, 31, 9), (32, 32, 32), (64, 64, 17), (65, 63, 33), (63, 66, 31), (66, 2, 130), (1, 129, 65),
         (96, 33, 47), (257, 34, 16), (700, 3, 5)]


def _embed(dmrg_amd, a, dtype, off, pad):
    """Device address of `a` inside a NaN-filled array, its leading dimension and the owner."""
    rows, cols = a.shape
    ld = rows + pad
    flat = np.full(off + ld * cols + 8, np.nan, dtype=dtype)
    for j in range(cols):
        flat[off + j * ld: off + j * ld + rows] = a[:, j]
    dev = dmrg_amd.DeviceArray.from_numpy(flat)
    return ctypes.c_void_p(dev.ptr.value + off * flat.itemsize), ld, dev


def _run(dmrg_amd, ops, dtype, opA, opB, M, N, K, off, pad, beta):
    cplx = dtype == np.complex128
    rng = np.random.default_rng(M + 100 * N + 10000 * K + opA + 4 * opB)
    A = rand(rng, (K, M) if opA in (1, 3) else (M, K), cplx).astype(dtype)
    B = rand(rng, (N, K) if opB in (1, 3) else (K, N), cplx).astype(dtype)
    C = rand(rng, (M, N), cplx).astype(dtype)
    f = {0: lambda x: x, 1: lambda x: x.T, 2: lambda x: x.conj(), 3: lambda x: x.conj().T}
    wide = np.complex128 if cplx else np.float64
    ref = f[opA](A).astype(wide) @ f[opB](B).astype(wide) + beta * C.astype(wide)
    pa, lda, ka = _embed(dmrg_amd, A, dtype, off, pad)
    pb, ldb, kb = _embed(dmrg_amd, B, dtype, off + 1, pad + 2)
    pc, ldc, kc = _embed(dmrg_amd, C, dtype, off, pad)
    lib = dmrg_amd.lib()
    if dtype == np.float32:
        rc = lib.dmrg_op_gemm_f32(ops._h, None, dmrg_amd.PREC_FP32, opA, opB, M, N, K, pa, lda, pb, ldb, pc, ldc)
    else:
        one, be = np.array([1], dtype), np.array([beta], dtype)
        rc = lib.dmrg_op_gemm(ops._h, None, 1 if cplx else 0, opA, opB, M, N, K, one.ctypes.data, pa, lda, pb, ldb,
                              be.ctypes.data, pc, ldc)
    assert rc == dmrg_amd.OK, lib.dmrg_last_error()
    out = kc.numpy()
    got = np.stack([out[off + j * ldc: off + j * ldc + M] for j in range(N)], axis=1)
    out[np.concatenate([np.arange(off + j * ldc, off + j * ldc + M) for j in range(N)])] = np.nan
    assert np.isnan(out).all()  # nothing written outside C
    return rel_err(got.astype(wide), ref)


@pytest.mark.parametrize("shape", EDGES)
def test_edges(dmrg_amd, ops, shape):
    for off, pad in ((0, 0), (1, 1), (3, 2)):
        for opA, opB in ((0, 0), (1, 0), (0, 1), (1, 1)):
            assert _run(dmrg_amd, ops, np.float64, opA, opB, *shape, off, pad, 0.5) < 1e-13, (off, opA, opB)
            assert _run(dmrg_amd, ops, np.float32, opA, opB, *shape, off, pad, 0.0) < 1e-5, (off, opA, opB)
        for opA, opB in ((0, 0), (3, 0), (0, 3), (2, 1), (1, 2), (3, 3)):
            assert _run(dmrg_amd, ops, np.complex128, opA, opB, *shape, off, pad, 0.5) < 1e-13, (off, opA, opB)


@pytest.mark.parametrize("cL,cR,D", [(1, 1, 5), (2, 90, 11), (33, 65, 5), (70, 150, 11), (40, 129, 7)])
def test_sliced_sums(dmrg_amd, ops, cL, cR, D):
    """K-heavy products whose k is cut into slices: the out-step of the
    matvecs (K = D cR, odd and even) and of both environment updates."""
    rng = np.random.default_rng(cL + cR + D)
    L, R, W = rand(rng, (cL, D, cL), False), rand(rng, (cR, D, cR), False), rand(rng, (D, 2, 2, D), False)
    dev = dmrg_amd.DeviceArray.from_numpy
    th1, th2 = rand(rng, (cL, 2, cR), False), rand(rng, (cL, 2, 2, cR), False)
    o1, o2 = (dmrg_amd.DeviceArray(x.shape, x.dtype) for x in (th1, th2))
    ops.heff1(dev(L), dev(R), dev(W), dev(th1), o1)
    assert rel_err(o1.numpy(), od.apply_heff1(L, R, W, th1)) < 1e-12
    ops.heff2(dev(L), dev(R), dev(W), dev(W), dev(th2), o2)
    assert rel_err(o2.numpy(), od.apply_heff2(L, R, W, W, th2)) < 1e-12
    f32 = lambda x: dev(x.astype(np.float32), np.float32)  # noqa: E731
    o3 = dmrg_amd.DeviceArray(th2.shape, np.float32)
    ops.heff2_f32(f32(L), f32(R), dev(W), dev(W), f32(th2), o3)
    assert rel_err(o3.numpy().astype(np.float64), od.apply_heff2(L, R, W, W, th2)) < 2e-5
    A, B = rand(rng, (cR, 2, cL), False), rand(rng, (cL, 2, cR), False)
    l, r = (dmrg_amd.DeviceArray((cL, D, cL), np.float64) for _ in range(2))
    ops.env_left(dev(R), dev(A), dev(W), l)
    assert rel_err(l.numpy(), od.update_left_env(R, A, W)) < 1e-12
    ops.env_right(dev(R), dev(B), dev(W), r)
    assert rel_err(r.numpy(), od.update_right_env(R, B, W)) < 1e-12
