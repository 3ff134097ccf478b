"""Tuning a GEMM shape while another thread captures a stream: neither the call
nor the capture may fail (draining the device would make both)."""
import ctypes as C
import threading

import numpy as np
import pytest

from conftest import rand, rel_err

pytestmark = pytest.mark.gpu


def test_tuner_during_a_capture(dmrg_amd, ops):
    lib, rng = dmrg_amd.lib(), np.random.default_rng(1)
    A, B = rand(rng, (83, 71)), rand(rng, (71, 93))  # a shape that no other test uses
    dA, dB = (dmrg_amd.DeviceArray.from_numpy(x) for x in (A, B))
    out = [dmrg_amd.DeviceArray((83, 93), np.float64) for _ in range(2)]
    with dmrg_amd.DMRG(4, 2, 4, 5, autotune=1) as eng:  # switches the tuner on
        tuned = eng.stats()["tuned_shapes"]
        s, g = C.c_void_p(), C.c_void_p()
        assert lib.hipStreamCreateWithFlags(C.byref(s), 1) == 0
        assert lib.hipStreamBeginCapture(s, 1) == 0  # thread-local mode
        err = []

        def call():
            try:
                ops.gemm(0, 0, dA, dB, out[0])
            except Exception as e:  # noqa: BLE001
                err.append(e)

        t = threading.Thread(target=call)
        t.start()
        t.join()
        assert lib.hipStreamEndCapture(s, C.byref(g)) == 0
        assert not err, err
        assert eng.stats()["tuned_shapes"] == tuned + 1
        ops.gemm(0, 0, dA, dB, out[1])
        assert eng.stats()["tuned_shapes"] == tuned + 1
    assert rel_err(out[0].numpy(), A @ B) < 1e-13
    assert np.array_equal(out[0].numpy(), out[1].numpy())
    assert lib.hipGraphDestroy(g) == 0 and lib.hipStreamDestroy(s) == 0
