"""Parity of the staggered (MAC) scheme's HIP path against the FP64 oracle's
restatement of PML_WaveSolver::stepLeapfrog (src/wavesolver/PML_WaveSolver.cpp:
710-773) on seeded free-field scenes.

Tolerance: listener relative L2 error <= 1e-4 over the whole time series and
pressure-field relative L2 error <= 1e-4 at the end; every tile plan gives
the same fields bit for bit."""
import numpy as np
import pytest

from acoustics_amd import scenes
from acoustics_amd.solver import Solver, rel_l2
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-4


def test_staggered_free_field_matches_oracle(hip_lib):
    sb, steps = scenes.staggered_free_field(seed=7, div=(40, 44, 36), pml=6, steps=300)
    print(f"case: staggered divisions={sb.divisions} steps={steps}", flush=True)
    o = Oracle(sb, reclassify_each_step=False)
    ref = o.step(steps)
    p_ref = o.pressure()
    o.close()
    with Solver(sb) as s:
        s.step(steps)
        got = s.series()
        p_got = s.pressure()
    assert np.all(np.isfinite(got))
    err = rel_l2(got, ref)
    errp = rel_l2(p_got, p_ref)
    print("staggered listener rel L2", err, "field rel L2", errp)
    assert err <= TOL
    assert errp <= TOL


def test_staggered_tile_plans_agree(hip_lib):
    sb, _ = scenes.staggered_free_field(seed=8, div=(32, 32, 40), pml=5)
    print(f"case: staggered plans divisions={sb.divisions}", flush=True)
    base = None
    for plan in range(11):
        with Solver(sb, tile_config=plan) as s:
            s.step(120)
            out = (s.series(), s.pressure())
        if base is None:
            base = out
        else:
            assert np.array_equal(out[0], base[0]), plan
            assert np.array_equal(out[1], base[1]), plan


def test_staggered_float4_rows_carry_listeners(hip_lib):
    """Rows long enough for the float4 row tiles (the default plan), with
    listeners whose MLS cells lie in them: every plan gives the same series
    bit for bit and the oracle's to 1e-4 (a row tile that dropped its cells'
    listener terms lost part of each listener's sum)."""
    sb, steps = scenes.staggered_free_field(seed=9, div=(72, 64, 80), pml=6, steps=200, n_listeners=12)
    print(f"case: staggered float4 rows divisions={sb.divisions} steps={steps}", flush=True)
    ref = Oracle(sb, reclassify_each_step=False).step(steps)
    outs = []
    for plan in (3, 4, 8):
        with Solver(sb, tile_config=plan) as s:
            s.step(steps)
            outs.append(s.series())
    for o in outs[1:]:
        assert np.array_equal(o, outs[0])
    assert rel_l2(outs[0], ref) <= TOL


def test_rows_past_the_caches(hip_lib):
    """A grid of just over nine million cells, whose float4 rows are stored past
    the caches: ragged rows, the same bits as the scalar tiles, fused or not."""
    sb, _ = scenes.staggered_free_field(seed=10, div=(206, 211, 209), pml=6, n_listeners=8)
    print(f"case: staggered rows past the caches divisions={sb.divisions}", flush=True)
    base = None
    for plan in (8, -1, 1, 3):
        with Solver(sb, tile_config=plan) as s:
            s.step(60)
            out = (s.series(), s.pressure())
        if base is None:
            base = out
            assert np.abs(out[1]).max() > 0
        else:
            assert np.array_equal(out[0], base[0]), plan
            assert np.array_equal(out[1], base[1]), plan
