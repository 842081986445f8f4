"""Rows longer than a wavefront's 256 cells run as float4 row segments: the
same bits as the scalar tiles (plan 4), at segment edges and remainders, with
listeners around the cuts."""
import numpy as np
import pytest

from acoustics_amd import capi, scenes
from acoustics_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [272, 273, 276, 333, 531])
@pytest.mark.parametrize("scheme", [capi.FDTD_SCHEME_COLLOCATED, capi.FDTD_SCHEME_STAGGERED])
def test_segments_match_scalar_tiles(hip_lib, nz, scheme):
    s = scenes.base_settings((20, 22, nz), 0.005, 5)
    s["scheme"] = scheme
    h, mb = 0.005, np.array(s["min_bound"])
    # a pulse of a few cells away from the rows' middle, listeners along the rows
    src = scenes.gaussian_pressure_source(mb + h * np.array([10.2, 9.8, 0.3 * nz]), 2e-5)
    ears = mb + h * np.stack([np.full(24, 9.6), np.full(24, 12.3), np.linspace(0.2 * nz, 0.9 * nz, 24)], axis=1)
    sb = scenes.SceneBuffers(s, pressure_sources=[src], listeners=ears)
    print(f"case: long rows {nz} scheme {scheme}", flush=True)
    out = []
    states = (capi.FDTD_PML_STATE_MERGED, capi.FDTD_PML_STATE_SPLIT) if scheme else (capi.FDTD_PML_STATE_MERGED,)
    for state in states:
        for plan in (0, 1, 4):
            with Solver(sb, tile_config=plan, pml_state=state) as v:
                v.step(160)
                out.append((v.series(), v.pressure()))
        assert np.abs(out[-1][0]).max() > 0
        for o in out[1:]:
            assert np.array_equal(o[0], out[0][0]) and np.array_equal(o[1], out[0][1])
        out.clear()
