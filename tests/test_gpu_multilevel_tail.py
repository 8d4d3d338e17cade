"""The single-workgroup kernel of the multilevel cycle's small levels, at the
shapes where its aggregates end: one cycle (FP32) of a grid that starts in it,
or whose second or third level does, against the float64 restatement of
tests/mg_reference.py. FP32 rounding (6e-8) of some 20 dependent operations per site
and level over six levels is within 1e-5 of the largest entry; a wrong
neighbour or coupling is 1e-3 or more."""
from __future__ import annotations

import numpy as np
import pytest

import microsimulator_amd as msa

from tests.test_gpu_flow import _multilevel_reference, grids, random_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    (16, 16), (5, 3),                     # the dense inverse alone
    (17, 16), (2, 129), (33, 9),          # one level above it, odd remainders
    (64, 64), (63, 65), (32, 128),        # the most cells and aggregates it takes
    (2, 2047), (2048, 2), (3, 1365),      # thin: many aggregates for the cells
    (65, 64), (129, 127), (1, 3000),      # one more level on the tiles
    (515, 259),                           # three
])
def test_cycle_at_the_tails_edges(hip, oracle, shape):
    nx, ny = shape
    thin = min(shape) < 5
    solid, mob = random_case(17, nx, ny, solid_fraction=0.0 if thin else 0.1)
    g, og = grids(nx, ny, 1.0, solid, dx=1.25, dy=0.75)
    hip.flow_prepare(g, mob, 0)
    ml = _multilevel_reference(oracle, og, mob, nx, ny, 1.25, 0.75)
    r = np.random.default_rng(3).standard_normal(nx * ny).astype(np.float32)
    r[solid != 0] = 0.0
    z = hip.flow_precondition(r).astype(np.float64)
    ref = ml.cycle(r.astype(np.float64).reshape(nx, ny)).ravel()
    err = np.abs(z - ref).max() / np.abs(ref).max()
    print(shape, "levels", len(ml.levels), "relative error", err, flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("shape", [(64, 64), (63, 65), (129, 127), (515, 259)])
@pytest.mark.parametrize("lds", [0, 6000, 64 << 10, 80 << 10])
def test_cycle_with_less_lds(oracle, shape, lds):
    """The same cycle where a workgroup has less LDS than the tail would take:
    it starts at a smaller level, at the latest the coarsest."""
    nx, ny = shape
    solid, mob = random_case(17, nx, ny, solid_fraction=0.1)
    g, og = grids(nx, ny, 1.0, solid, dx=1.25, dy=0.75)
    ml = _multilevel_reference(oracle, og, mob, nx, ny, 1.25, 0.75)
    r = np.random.default_rng(3).standard_normal(nx * ny).astype(np.float32)
    r[solid != 0] = 0.0
    with msa.HipBackend(0) as hip:
        hip.set_resident_limits(lds_bytes=lds)
        hip.flow_prepare(g, mob, 0)
        z = hip.flow_precondition(r).astype(np.float64)
        rep = hip.flow_solve(msa.DepthAveragedFlowParameters(
            mean_inlet_speed=1.0, axis=0, relative_tolerance=1e-8, max_iterations=2000,
            solver=msa.SOLVER_MULTIGRID))
    ref = ml.cycle(r.astype(np.float64).reshape(nx, ny)).ravel()
    assert np.abs(z - ref).max() <= 1e-5 * np.abs(ref).max()
    assert rep.true_relative_residual <= 1e-8
