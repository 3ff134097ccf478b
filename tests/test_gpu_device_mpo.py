"""The operator calls derive their MPO matrices on the device, in stream order.

Each call is compared with the oracle for MPO sizes from the smallest on (the
derived matrix has (D d^2)^2 or (D d)^2 entries, one thread each, 256 to a
workgroup), and two calls in a row with different MPOs share one buffer.
Tolerance: as for the operators themselves, 1e-12 relative (FP64 sums of at
most D d^2 max(cL, cR) terms of order one); FP32: 2e-5 (three FP32 stages).
"""
import numpy as np
import pytest

from conftest import rand, rel_err
from oracle import dmrg as od

pytestmark = pytest.mark.gpu


def _dev(dmrg_amd, *arrays):
    return [dmrg_amd.DeviceArray.from_numpy(a) for a in arrays]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("d,D", [(1, 1), (2, 1), (1, 3), (3, 2), (2, 11), (4, 8)])
def test_two_site_mpo(dmrg_amd, ops, cplx, d, D):
    rng = np.random.default_rng(100 * d + D)
    cL, cR = 3, 5
    L, R = rand(rng, (cL, D, cL), cplx), rand(rng, (cR, D, cR), cplx)
    th = rand(rng, (cL, d, d, cR), cplx)
    W = [rand(rng, (D, d, d, D), cplx) for _ in range(3)]
    dL, dR, dth, *dW = _dev(dmrg_amd, L, R, th, *W)
    outs = [dmrg_amd.DeviceArray(th.shape, th.dtype) for _ in range(2)]
    for i, out in enumerate(outs):  # the second call's matrix follows the first call's product
        ops.heff2(dL, dR, dW[i], dW[i + 1], dth, out)
    for i, out in enumerate(outs):
        assert rel_err(out.numpy(), od.apply_heff2(L, R, W[i], W[i + 1], th)) < 1e-12


@pytest.mark.parametrize("d,D", [(1, 1), (2, 11), (4, 8)])
def test_two_site_mpo_f32(dmrg_amd, ops, d, D):
    rng = np.random.default_rng(200 * d + D)
    cL, cR = 6, 4
    L, R = (rand(rng, (c, D, c), False).astype(np.float32) for c in (cL, cR))
    th = rand(rng, (cL, d, d, cR), False).astype(np.float32)
    W1, W2 = (rand(rng, (D, d, d, D), False) for _ in range(2))
    out = dmrg_amd.DeviceArray(th.shape, np.float32)
    ops.heff2_f32(*_dev(dmrg_amd, L, R, W1, W2, th), out)
    ref = od.apply_heff2(*(x.astype(np.float64) for x in (L, R, W1, W2, th)))
    assert rel_err(out.numpy().astype(np.float64), ref) < 2e-5


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("d,D", [(1, 1), (3, 2), (2, 11), (5, 4)])
def test_right_environment_mpo(dmrg_amd, ops, cplx, d, D):
    rng = np.random.default_rng(300 * d + D)
    ci, co = 4, 6
    R, A = rand(rng, (ci, D, ci), cplx), rand(rng, (co, d, ci), cplx)
    W = rand(rng, (D, d, d, D), cplx)
    out = dmrg_amd.DeviceArray((co, D, co), A.dtype)
    ops.env_right(*_dev(dmrg_amd, R, A, W), out)
    assert rel_err(out.numpy(), od.update_right_env(R, A, W)) < 1e-12
