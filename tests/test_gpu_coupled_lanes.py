"""Coupled ghosts whose operator rows are shared by lanes give the oracle's
signals."""
import pytest

from acoustics_amd import capi, scenes
from acoustics_amd.solver import Solver, rel_l2
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_obj", [1, 3])
def test_against_oracle(hip_lib, n_obj):
    sb, _ = scenes.config3(seed=11, n=60, h=0.005, pml=6, n_obj=n_obj, n_listeners=16, axis_lo=0.012, axis_hi=0.03,
                           boundary=capi.FDTD_BOUNDARY_FULLY_COUPLED)
    ref = Oracle(sb, reclassify_each_step=False).step(200)
    with Solver(sb) as s:
        s.step(200)
        got = s.series()
    assert rel_l2(got, ref) <= 1e-4
