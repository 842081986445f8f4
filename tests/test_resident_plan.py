"""Host check of the cut of scenes that run resident (fdtd_plan_check covers
it with the tile plans): every cell, object-adjacent record and listener term
in exactly one tile of its class, within what a workgroup holds."""
import ctypes as C

import numpy as np
import pytest

from acoustics_amd import capi, scenes


def _check(sb):
    lib = capi.load_library()
    capi.check(lib.fdtd_plan_check(sb.ref(), 0, None), "fdtd_plan_check")


@pytest.mark.parametrize("div,pml", [((18, 17, 19), 6), ((24, 14, 40), 3), ((37, 29, 41), 2), ((20, 24, 300), 5),
                                     ((260, 22, 21), 5), ((70, 71, 72), 16), ((64, 64, 64), 10), ((21, 400, 23), 7)])
def test_free_field(div, pml):
    s = scenes.base_settings(div, 0.005, pml)
    lo, hi = scenes.interior_bounds(s, 1)
    rng = np.random.default_rng(1)
    full = np.array(s["min_bound"]) + 0.005 * np.array(div) * rng.uniform(0.02, 0.98, size=(20, 3))
    _check(scenes.SceneBuffers(s, pressure_sources=[scenes.gaussian_pressure_source(0.5 * (lo + hi), 1e-4)], listeners=full))


@pytest.mark.parametrize("seed", range(4))
def test_objects(seed):
    _check(scenes.config2(seed=seed, n=64, n_listeners=24, radius=0.03, shell=0.045)[0])
    for sb in scenes.config4(seed=seed, n_scenes=3, edge_lo=24, edge_hi=90)[0]:
        _check(sb)
    _check(scenes.vibration_scene(seed=seed)[0])


@pytest.mark.parametrize("width", [2.5, 6.5, 7.999])
def test_fractional_pml_widths(width):
    """A PML that ends inside a cell: the scene is cut or left to the step
    kernels, never cut wrongly."""
    s = scenes.base_settings((40, 36, 44), 0.005, 8)
    s["pml_width"] = width
    _check(scenes.SceneBuffers(s, listeners=np.zeros((1, 3))))
