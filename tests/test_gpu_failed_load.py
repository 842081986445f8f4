"""A snapshot that cannot be loaded (a file missing or short) leaves the handle
as it was: the same signals and field as one that never tried, bit for bit."""
import os

import numpy as np
import pytest

from acoustics_amd import capi, scenes
from acoustics_amd.solver import Solver

pytestmark = pytest.mark.gpu


def _scene(scheme):
    s = scenes.base_settings((36, 32, 40), 0.005, 6)
    s["scheme"] = scheme
    return scenes.SceneBuffers(s, pressure_sources=[scenes.gaussian_pressure_source(np.array([0.004, -0.003, 0.01]), 5e-5)],
                               listeners=np.random.default_rng(3).uniform(-0.04, 0.04, size=(6, 3)))


@pytest.mark.parametrize("scheme", [capi.FDTD_SCHEME_COLLOCATED, capi.FDTD_SCHEME_STAGGERED])
def test_a_failed_load_changes_nothing(hip_lib, tmp_path, scheme):
    sb = _scene(scheme)
    pat = str(tmp_path / "s_%s")
    with Solver(sb, pml_state=capi.FDTD_PML_STATE_SPLIT) as a:
        a.step(30)
        a.save_snapshot(pat, "0", 1)
    with Solver(sb) as a:
        a.step(150)
        want, field = a.series(), a.pressure()
    os.remove(str(tmp_path / "s_0_snapshot_1_engine_state.bin"))
    with Solver(sb) as b:
        b.step(90)
        with pytest.raises(RuntimeError):
            b.load_snapshot(str(tmp_path / "none_%s"), "0", 1)
        for last in ("v_pml_2.dat", "p_pml_1.dat", "step.txt"):     # ever earlier files missing
            os.remove(str(tmp_path / ("s_0_snapshot_1_" + last)))
            with pytest.raises(RuntimeError):
                b.load_snapshot(pat, "0", 1)
        b.step(60)
        assert np.array_equal(b.series(), want)
        assert np.array_equal(b.pressure(), field)
