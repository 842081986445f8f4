"""Handles and batches on streams that their caller captures: what is recorded
gives the eager signals on its replays, and another handle's blocks, which the
recording must not catch, run meanwhile."""
import ctypes as C

import numpy as np
import pytest

from acoustics_amd import capi, scenes
from acoustics_amd.solver import Batch, Solver

pytestmark = pytest.mark.gpu

CAPTURE_RELAXED = 2


class Stream:
    def __init__(self):
        self.hip = C.CDLL("libamdhip64.so.7")
        self.s = C.c_void_p()
        assert self.hip.hipStreamCreateWithFlags(C.byref(self.s), 1) == 0

    def begin(self):
        assert self.hip.hipStreamBeginCapture(self.s, CAPTURE_RELAXED) == 0

    def end(self):
        g, self.x = C.c_void_p(), C.c_void_p()
        assert self.hip.hipStreamEndCapture(self.s, C.byref(g)) == 0
        assert self.hip.hipGraphInstantiate(C.byref(self.x), g, None, None, 0) == 0

    def replay(self):
        assert self.hip.hipGraphLaunch(self.x, self.s) == 0
        assert self.hip.hipStreamSynchronize(self.s) == 0


class StreamBatch(Batch):
    """A batch on a caller's stream."""

    def __init__(self, sbs, steps, stream):
        self.lib, self.sbs, self.steps = capi.load_library(), list(sbs), list(steps)
        self._arr = (capi.Scene * len(sbs))(*[sb.scene for sb in sbs])
        opt = capi.BatchOptions()
        self.lib.fdtd_batch_options_default(C.byref(opt))
        opt.stream = stream.s.value
        self.h = C.c_void_p()
        capi.check(self.lib.fdtd_batch_create(self._arr, (C.c_int * len(steps))(*steps), len(sbs), C.byref(opt),
                                              C.byref(self.h)), "fdtd_batch_create")


def _sphere(n, seed=2):
    return scenes.config2(seed=seed, n=n, n_listeners=12, radius=0.03, shell=0.045)[0]


def test_a_block_beside_a_captured_one(hip_lib):
    sb = _sphere(64)
    with Solver(sb, tile_config=0) as s:
        s.step(196)
        want, field = s.series(), s.pressure()
    st = Stream()
    with Solver(sb, stream=st.s.value) as a, Solver(sb) as b:
        print("case: capture beside a resident block", flush=True)
        a.step(64)                      # resident
        st.begin()
        a.step(66)                      # recorded
        b.step(130)                     # resident, meanwhile
        b.synchronize()
        st.end()
        assert np.array_equal(b.series(), want[:130])
        st.replay()
        assert np.array_equal(a.series(), want[:130])
        a.step(66)                      # resident again
        assert np.array_equal(a.series(), want) and np.array_equal(a.pressure(), field)


@pytest.mark.parametrize("block", [20, 70])
def test_a_captured_batch(hip_lib, block):
    sbs = [_sphere(56), _sphere(64, 3)]
    steps = [300, 280]
    with Batch(sbs, steps, tile_config=0) as b:
        b.run()
        want = [b.series(i) for i in range(2)]
    st = Stream()
    with StreamBatch(sbs, steps, st) as b:
        print(f"case: captured batch, blocks of {block}", flush=True)
        b.step(64)
        st.begin()
        b.step(block)
        st.end()
        st.replay()
        assert all(np.array_equal(b.series(i), want[i][:64 + block]) for i in range(2))
        b.run()
        assert all(np.array_equal(b.series(i), want[i]) for i in range(2))
