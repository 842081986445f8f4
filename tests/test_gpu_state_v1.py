"""Engine state files of version 1, which hold a merged PML by its six slabs,
resume bit for bit: a file written when that was the engine's own storage, with
the signals and the field 30 steps later."""
import os

import numpy as np
import pytest

from acoustics_amd import capi, scenes
from acoustics_amd.solver import Solver

pytestmark = pytest.mark.gpu


def test_version_1_state_resumes(hip_lib, tmp_path):
    old = np.load(os.path.join(os.path.dirname(__file__), "data", "engine_state_v1.npz"))
    s = scenes.base_settings((14, 12, 13), 0.005, 3.0)
    mid = np.array(s["min_bound"]) + 0.005 * np.array([7.2, 6.4, 6.1])
    sb = scenes.SceneBuffers(s, pressure_sources=[scenes.gaussian_pressure_source(mid, 2e-5)],
                             listeners=np.array([mid + 0.008, mid - 0.007]))
    (tmp_path / "r_x_snapshot_0_engine_state.bin").write_bytes(old["state"].tobytes())
    for kw in (dict(tile_config=0), dict()):
        with Solver(sb, **kw) as v:
            v.load_snapshot(str(tmp_path / "r_%s"), "x", 0)
            v.step(30)
            assert np.array_equal(v.series(41, 30), old["series"])
            assert np.array_equal(v.pressure().astype(np.float32), old["pressure"])
            # and so does the file that this handle writes
            v.save_snapshot(str(tmp_path / "n_%s"), "x", 0)
            v.step(20)
            want = v.series(71, 20)
        with Solver(sb, **kw) as v:
            v.load_snapshot(str(tmp_path / "n_%s"), "x", 0)
            v.step(20)
            assert np.array_equal(v.series(71, 20), want)
    # a split handle refuses it as before
    with Solver(sb, pml_state=capi.FDTD_PML_STATE_SPLIT) as v, pytest.raises(RuntimeError):
        v.load_snapshot(str(tmp_path / "r_%s"), "x", 0)
