"""Scenes held on the chip for a block of steps (resident.hip): the same bits
as the step kernels, at the edges of its tiles (grids from one tile to the
largest that fits, edges off every tile size, each PML depth), with sources,
objects, listeners and both object samplings, over blocks of any length mixed
with single steps, in batches, beside another thread, and when a launch gives
its block up."""
import threading

import numpy as np
import pytest

from acoustics_amd import capi, scenes
from acoustics_amd.solver import Batch, Server, Solver

pytestmark = pytest.mark.gpu


def _free(div, pml, seed=3):
    rng = np.random.default_rng(seed)
    s = scenes.base_settings(div, 0.005, pml)
    lo, hi = scenes.interior_bounds(s, 1)
    mid = 0.5 * (lo + hi)
    src = [scenes.gaussian_pressure_source(mid + 0.3 * (hi - mid) * rng.uniform(-1, 1, 3), 4e-5) for _ in range(2)]
    full = np.array(s["min_bound"])
    span = 0.005 * np.array(div)
    # listeners in the interior and anywhere in the PML
    ears = np.vstack([rng.uniform(lo, hi, size=(4, 3)), full + span * rng.uniform(0.02, 0.98, size=(12, 3))])
    return scenes.SceneBuffers(s, pressure_sources=src, listeners=ears)


CASES = {
    "one_tile_boxes": lambda: _free((18, 17, 19), 6),
    "thin_interior": lambda: _free((24, 8 + 2 * 3, 40), 3),
    "two_layer_pml": lambda: _free((37, 29, 41), 2),
    "odd": lambda: _free((33, 50, 65), 7),
    "tile_multiples": lambda: _free((48, 48, 48), 8),
    "deep_pml": lambda: _free((70, 71, 72), 16),
    "long": lambda: _free((20, 24, 300), 5),
    "wide": lambda: _free((260, 22, 21), 5),
    "sphere": lambda: scenes.config2(seed=2, n=64, n_listeners=24, radius=0.03, shell=0.045)[0],
    "sphere_seven": lambda: scenes.with_settings(scenes.config2(seed=4, n=64, n_listeners=24, radius=0.03, shell=0.045)[0],
                                                 sampling=capi.FDTD_SAMPLE_SEVEN),
    "ellipsoids": lambda: scenes.vibration_scene(seed=5, n=56, acc_noise=False, gaussian=True, chirp=True)[0],
    "largest": lambda: scenes.config2(seed=2)[0],
}


@pytest.mark.parametrize("name", list(CASES))
def test_same_bits_as_the_step_kernels(hip_lib, name):
    sb = CASES[name]()
    print(f"case: resident {name} {sb.divisions}", flush=True)
    with Solver(sb, tile_config=0) as a, Solver(sb) as b:
        # single steps, blocks below and above a launch's 64, and their mixtures
        for n in (1, 5, 64, 3, 130, 2, 9):
            a.step(n)
            b.step(n)
            assert np.array_equal(a.pressure(), b.pressure()), n
        assert np.abs(a.series()).max() > 0
        assert np.array_equal(a.series(), b.series())


def test_blocks_wrap_the_series_ring(hip_lib):
    sb = CASES["sphere"]()
    with Solver(sb, tile_config=0) as a, Solver(sb, series_capacity=50) as b:
        a.step(333)
        b.step(333)
        assert np.array_equal(a.series(), b.series())


def test_given_up_blocks_are_run_by_the_step_kernels(hip_lib, monkeypatch):
    """A wait limit of zero: the first workgroup to look finds the others
    missing and gives the block up (or finds them all there and runs)."""
    sbs = [CASES["odd"](), CASES["sphere"]()]
    ref = []
    for sb in sbs:
        with Solver(sb, tile_config=0) as s:
            s.step(200)
            ref.append(s.series())
    monkeypatch.setenv("FDTD_RESIDENT_WAIT", "0")
    for sb, want in zip(sbs, ref):
        with Solver(sb) as s:
            s.step(70)
            s.listen()
            s.step(130)
            assert np.array_equal(s.series(), want)
    with Batch(sbs, [200, 200]) as b:
        b.run()
        assert all(np.array_equal(b.series(i), ref[i]) for i in range(2))
    with Server(steps_per_block=48) as srv:
        ids = [srv.submit(sb, 200) for sb in sbs]
        for rid, want in zip(ids, ref):
            assert srv.wait(rid, 60000) == 0
            assert np.array_equal(srv.take(rid)[1], want)


@pytest.mark.parametrize("name", ["odd", "sphere"])
def test_short_blocks_behind_a_given_up_one(hip_lib, monkeypatch, name):
    """Step kernels enqueued before the host knows of it leave the scene alone."""
    sb = CASES[name]()
    with Solver(sb, tile_config=0) as s:
        s.step(203)
        want = s.series()
    monkeypatch.setenv("FDTD_RESIDENT_WAIT", "0")
    with Solver(sb) as s:
        for n in (70, 2, 1, 127, 3):
            s.step(n)
        assert np.array_equal(s.series(), want)


def test_two_threads(hip_lib):
    """Two handles on two streams, each too large to share the device."""
    sb = CASES["largest"]()
    with Solver(sb, tile_config=0) as s:
        s.step(256)
        want = s.series()
    got = [None, None]

    def work(i):
        with Solver(sb) as s:
            for _ in range(4):
                s.step(64)
            got[i] = s.series()
    th = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert all(np.array_equal(g, want) for g in got)


def _large(kind, div):
    rng = np.random.default_rng(8)
    if kind == "staggered":
        s = scenes.base_settings(div, 0.005, 8)
        s["scheme"] = capi.FDTD_SCHEME_STAGGERED
        mid = np.array(s["min_bound"]) + 0.005 * np.array(div) * [0.5, 0.08, 0.5]   # the pulse reaches into the PML
        ears = mid + rng.uniform(0.0, 0.06, size=(12, 3))
        return scenes.SceneBuffers(s, pressure_sources=[scenes.gaussian_pressure_source(mid, 2e-5)], listeners=ears)
    return scenes._small_object_scene(rng, div, 0.005, 8, 2, 24)


@pytest.mark.parametrize("kind", ["objects", "staggered"])
@pytest.mark.parametrize("div", [(139, 89, 190), (144, 146, 144), (97, 210, 133)])
def test_grids_for_the_largest_tiles(hip_lib, kind, div):
    """Too many tiles of the other shapes: columns of up to 32 cells, along x and y, in one LDS buffer."""
    sb = _large(kind, div)
    print(f"case: large {kind} {div}", flush=True)
    with Solver(sb, tile_config=0) as s:
        s.step(150)
        want, field = s.series(), s.pressure()
        s.step(61)
        more = s.pressure()
    with Solver(sb) as s:
        for n in (1, 70, 79):
            s.step(n)
        assert np.array_equal(s.series(), want) and np.array_equal(s.pressure(), field)
        s.step(60)
        s.step(1)      # a step kernel goes on from the block's two levels
        assert np.array_equal(s.pressure(), more)
