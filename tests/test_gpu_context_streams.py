"""One operator context used on several streams: its buffers (the fused MPO, the
contraction intermediates) belong to one call at a time, so each call waits on
the device for the one before it, whatever stream that ran on.

Every output must be the one of the same call made alone, bit for bit.  Sizes
alternate between large and small, so that without the wait a small call would
overtake the large one and overwrite its intermediates.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import rand

pytestmark = pytest.mark.gpu


class _Stream:
    """A stream of the runtime that the engine library uses, not ordered with the default one."""

    def __init__(self, lib):
        self.lib, self.h = lib, C.c_void_p()
        assert lib.hipStreamCreateWithFlags(C.byref(self.h), 1) == 0

    def destroy(self):
        assert self.lib.hipStreamDestroy(self.h) == 0


def _problem(dmrg_amd, rng, c, D):
    dev = dmrg_amd.DeviceArray.from_numpy
    L, R = (dev(rand(rng, (c, D, c))) for _ in range(2))
    W1, W2 = (dev(rand(rng, (D, 2, 2, D))) for _ in range(2))
    th, s = dev(rand(rng, (c, 2, 2, c))), dev(rand(rng, (c, 2, c)))
    f = [dev(rand(rng, sh).astype(np.float32)) for sh in ((c, D, c), (c, D, c), (c, 2, 2, c))]
    new = lambda shape, dt=np.float64: dmrg_amd.DeviceArray(shape, dt)
    return [
        (lambda o, out, st: o.heff2(L, R, W1, W2, th, out, stream=st), lambda: new((c, 2, 2, c))),
        (lambda o, out, st: o.heff1(L, R, W1, s, out, stream=st), lambda: new((c, 2, c))),
        (lambda o, out, st: o.env_right(R, s, W2, out, stream=st), lambda: new((c, D, c))),
        (lambda o, out, st: o.env_left(L, s, W2, out, stream=st), lambda: new((c, D, c))),
        (lambda o, out, st: o.heff2_f32(f[0], f[1], W1, W2, f[2], out, stream=st), lambda: new((c, 2, 2, c), np.float32)),
    ]


def test_calls_on_several_streams(dmrg_amd):
    rng = np.random.default_rng(11)
    sizes = [(300, 11), (12, 3), (200, 5), (9, 11)]
    probs = [_problem(dmrg_amd, rng, c, D) for c, D in sizes]
    alone = dmrg_amd.Ops(0)
    ref = []
    for p in probs:
        for call, out in p:
            o = out()
            call(alone, o, None)
            ref.append(o.numpy())
    lib = dmrg_amd.lib()
    streams = [_Stream(lib), _Stream(lib)]
    shared = dmrg_amd.Ops(0)
    for rep in range(4):
        got, order = [], [None, streams[0].h, streams[1].h, streams[0].h, None, streams[1].h, streams[1].h]
        outs = [out() for p in probs for _, out in p]
        n = 0
        for q in range(5):  # large and small in turn
            for i, p in enumerate(probs):
                p[q][0](shared, outs[5 * i + q], order[(n + rep) % len(order)])
                n += 1
                if rep == 2 and n == 7:  # a stream that goes, with work of the context pending
                    streams[0].destroy()
                    streams[0] = _Stream(lib)
                    order = [streams[0].h if s is order[1] or s is order[3] else s for s in order]
        dmrg_amd.synchronize()
        got = [o.numpy() for o in outs]
        assert all(np.array_equal(a, b) for a, b in zip(got, ref)), rep
    for s in streams:
        s.destroy()
    shared.close()
    alone.close()


def test_captured_call(dmrg_amd):
    """A call on a context whose buffers are large enough can be captured; the
    graph gives the call's result on every replay, between eager calls."""
    rng = np.random.default_rng(12)
    (heff2, out), other = _problem(dmrg_amd, rng, 64, 5)[0], _problem(dmrg_amd, rng, 40, 5)[0]
    lib, o = dmrg_amd.lib(), dmrg_amd.Ops(0)
    s = _Stream(lib)
    a, b, x = out(), out(), other[1]()
    heff2(o, a, None)
    other[0](o, x, s.h)
    dmrg_amd.synchronize()
    ref, ref_x = a.numpy(), x.numpy()
    g, ge = C.c_void_p(), C.c_void_p()
    assert lib.hipStreamBeginCapture(s.h, 0) == 0
    heff2(o, b, s.h)
    assert lib.hipStreamEndCapture(s.h, C.byref(g)) == 0
    assert lib.hipGraphInstantiate(C.byref(ge), g, None, None, C.c_size_t(0)) == 0
    for _ in range(3):
        dmrg_amd.copy_device(b, dmrg_amd.DeviceArray.from_numpy(np.zeros_like(ref)))
        assert lib.hipGraphLaunch(ge, s.h) == 0
        dmrg_amd.synchronize()
        assert np.array_equal(b.numpy(), ref)
        other[0](o, x, None)
        dmrg_amd.synchronize()
        assert np.array_equal(x.numpy(), ref_x)
    assert lib.hipGraphExecDestroy(ge) == 0 and lib.hipGraphDestroy(g) == 0
    s.destroy()
    o.close()
