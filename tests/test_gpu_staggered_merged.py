"""The staggered scheme's merged state (the increment of the pressure outside
the PML, the collocated merged state inside it): the oracle's signals to the
contract's 1e-4, the same bits from every tile plan and from resident blocks,
pulses that reach into the PML, and snapshots of handles that started merged."""
import filecmp
import os

import numpy as np
import pytest

from acoustics_amd import capi, scenes
from acoustics_amd.solver import Solver, rel_l2
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _scene(div, pml, edge=False, seed=5, width=6e-5):
    rng = np.random.default_rng(seed)
    s = scenes.base_settings(div, 0.005, pml)
    s["scheme"] = capi.FDTD_SCHEME_STAGGERED
    lo, hi = scenes.interior_bounds(s, 1)
    at = np.array([lo[0], hi[1], lo[2]]) if edge else rng.uniform(lo, hi)   # edge: next to three PML slabs
    src = [scenes.gaussian_pressure_source(at, width), scenes.gaussian_pressure_source(rng.uniform(lo, hi), width, offset=6 * width)]
    span = 0.005 * np.array(div)
    ears = np.vstack([rng.uniform(lo, hi, size=(6, 3)), np.array(s["min_bound"]) + span * rng.uniform(0.05, 0.95, size=(6, 3))])
    return scenes.SceneBuffers(s, pressure_sources=src, listeners=ears)


@pytest.mark.parametrize("div,pml,edge", [((32, 36, 40), 5, False), ((37, 29, 41), 4, True), ((66, 40, 51), 7, True),
                                          ((24, 50, 31), 2, False)])
def test_against_oracle_and_plans(hip_lib, div, pml, edge):
    sb = _scene(div, pml, edge)
    print(f"case: staggered merged {div} pml {pml} edge {edge}", flush=True)
    steps = 180
    ref = Oracle(sb, reclassify_each_step=False).step(steps)
    with Solver(sb) as s:
        s.step(3)                 # step kernels, then resident blocks
        s.step(steps - 3)
        got, field = s.series(), s.pressure()
    assert rel_l2(got, ref) <= 1e-4
    for plan in (0, 1, 4, 10):
        with Solver(sb, tile_config=plan) as s:
            s.step(steps)
            assert np.array_equal(s.series(), got), plan
            assert np.array_equal(s.pressure(), field), plan
    with Solver(sb, pml_state=capi.FDTD_PML_STATE_SPLIT) as s:
        s.step(steps)
        assert rel_l2(s.series(), got) <= 1e-5


@pytest.mark.parametrize("width", [5.3, 5.5, 5.7, 5.999])
def test_a_pml_that_ends_inside_a_cell(hip_lib, width):
    sb = _scene((36, 34, 40), 6)
    sb = scenes.with_settings(sb, pml_width=width)
    ref = Oracle(sb, reclassify_each_step=False).step(150)
    with Solver(sb) as s:
        s.step(150)
        assert rel_l2(s.series(), ref) <= 1e-4


def test_snapshots_of_a_handle_that_started_merged(hip_lib, tmp_path):
    sb = _scene((36, 32, 40), 6)
    pat, pat2 = str(tmp_path / "m_%s"), str(tmp_path / "s_%s")
    with Solver(sb) as a:
        a.step(90)
        a.save_snapshot(pat, "0", 1)
        rows = a.series()
        a.step(60)
        ser, field = a.series(), a.pressure()
    assert np.array_equal(ser[:90], rows)          # rows already read stay
    # the files are a split handle's, every one of them
    with Solver(sb, pml_state=capi.FDTD_PML_STATE_SPLIT) as b:
        b.step(90)
        b.save_snapshot(pat2, "0", 1)
    names = sorted(n for n in os.listdir(tmp_path) if n.startswith("m_"))
    assert len(names) >= 12
    for n in names:
        assert filecmp.cmp(tmp_path / n, tmp_path / ("s_" + n[2:]), shallow=False), n
    # a fresh default handle goes on from them bit for bit, with and without the engine's own file
    for drop in (False, True):
        if drop:
            os.remove(str(tmp_path / "m_0_snapshot_1_engine_state.bin"))
        with Solver(sb) as c:
            c.load_snapshot(pat, "0", 1)
            c.step(60)
            assert np.array_equal(c.series()[90:], ser[90:])
            assert np.array_equal(c.pressure(), field)
