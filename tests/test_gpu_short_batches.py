"""Batches stepped a few steps at a time (step kernels) and in longer calls
(resident blocks, in two tile shapes, beside a scene that is not resident): the
same bits as step kernels alone, also where blocks are given up."""
import numpy as np
import pytest

from acoustics_amd import scenes
from acoustics_amd.solver import Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wait", [None, "0"])
def test_short_and_long_calls(hip_lib, monkeypatch, wait):
    sbs = [scenes.config2(seed=2, n=64, n_listeners=12, radius=0.03, shell=0.045)[0],
           scenes._small_object_scene(np.random.default_rng(8), (144, 146, 144), 0.005, 8, 2, 12),     # the largest tiles
           scenes.moving_object(seed=10)[0]]                                                          # not resident
    steps = [300, 290, 40]
    with Batch(sbs, steps, tile_config=0) as b:
        b.run()
        want = [b.series(i) for i in range(3)]
    print(f"case: short and long batch calls, wait {wait}", flush=True)
    if wait is not None:
        monkeypatch.setenv("FDTD_RESIDENT_WAIT", wait)   # the first workgroup to look gives the block up
    with Batch(sbs, steps) as b:
        for n in (1, 2, 7, 60, 1, 3, 100, 5):
            b.step(n)
        assert np.array_equal(b.series(0), want[0][:179])
        b.run()
        for i in range(3):
            assert np.abs(want[i]).max() > 0
            assert np.array_equal(b.series(i), want[i]), i
