"""The fused first step of the two-site product (d = 2, real) for every MPO bond
that it serves, at the edges of its tiles of 16 rows and 16 columns.  FP64 1e-12,
FP32 2e-5, as for the operators themselves."""
import numpy as np
import pytest

from conftest import rand, rel_err
from oracle import dmrg as od

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", range(2, 9))
@pytest.mark.parametrize("cL,cR", [(1, 2), (3, 1), (15, 17), (16, 16), (17, 15), (33, 20), (50, 64)])
def test_all_mpo_bonds(dmrg_amd, ops, cL, cR, D):
    rng = np.random.default_rng(100 * D + cL)
    L, R, th = rand(rng, (cL, D, cL)), rand(rng, (cR, D, cR)), rand(rng, (cL, 2, 2, cR))
    W1, W2 = rand(rng, (D, 2, 2, D)), rand(rng, (D, 2, 2, D))
    ref = od.apply_heff2(L, R, W1, W2, th)
    dev = dmrg_amd.DeviceArray.from_numpy
    out = dmrg_amd.DeviceArray(th.shape, np.float64)
    ops.heff2(dev(L), dev(R), dev(W1), dev(W2), dev(th), out)
    assert rel_err(out.numpy(), ref) < 1e-12
    f32 = lambda x: dev(x.astype(np.float32))
    out = dmrg_amd.DeviceArray(th.shape, np.float32)
    ops.heff2_f32(f32(L), f32(R), dev(W1), dev(W2), f32(th), out)
    assert rel_err(out.numpy().astype(float), ref) < 2e-5
