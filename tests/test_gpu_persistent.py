"""Jacobi-PCG as one persistent launch (small and medium systems) against the
same iteration as two launches each, which a profiled solve takes.

Both stop on the same test of the same recurrence and differ in the order of
their FP64 sums only, so the iteration counts agree within the reference's own
allowance of 2 (tests/conformance/flow_conformance_test.cpp:259-263). Their
fields differ by what an iteration leaves at the stated residual, bounded for
these systems by 1e-5 of the largest speed as in the other solver-form tests.
"""
import numpy as np
import pytest

import microsimulator_amd as msa

pytestmark = pytest.mark.gpu

# Sites per workgroup are 512, 1024, 2048 or 4096 by the size; the halo is ny
# sites either side.
SHAPES = [
    (3, 2), (1, 7), (9, 1),          # one workgroup, most threads idle
    (16, 32), (19, 27), (27, 19),    # one whole workgroup; one site past it
    (64, 48), (131, 77),             # whole rows per workgroup; ragged
    (40, 700), (5, 1100),            # rows wider than a workgroup's sites
    (512, 256), (343, 383),          # 512 x 256 sites exactly; just past it
    (513, 511), (700, 751), (1023, 1025),
    (520, 2017), (300, 3600),        # more sites; halo past the LDS limit
]


def system(nx, ny, seed):
    rng = np.random.default_rng(seed)
    solid = np.zeros((nx, ny), np.uint8)
    if nx > 8 and ny > 8:
        for _ in range(max(1, nx * ny // 900)):
            x, y = rng.integers(2, nx - 4), rng.integers(1, ny - 4)
            solid[x:x + 3, y:y + 3] = 1
    mobility = rng.uniform(0.5, 2.0, (nx, ny)).astype(np.float32)
    return msa.Grid(nx, ny, 1, 1.0, 0.8, 10.0, solid), mobility


def solve(hip, solver, tolerance, profile, max_iterations=100000):
    rep = hip.flow_solve(msa.DepthAveragedFlowParameters(
        mean_inlet_speed=10.0, axis=0, relative_tolerance=tolerance, solver=solver,
        max_iterations=max_iterations, profile=profile))
    return rep, hip.flow_download()[1].concatenated()


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("solver", [msa.SOLVER_JACOBI_FP64, msa.SOLVER_MIXED])
def test_persistent_matches_launches(nx, ny, solver):
    grid, mobility = system(nx, ny, nx + ny)
    with msa.HipBackend(0) as hip:
        hip.flow_prepare(grid, mobility, 0)
        rep, faces = solve(hip, solver, 1e-8, False)
        ref, expected = solve(hip, solver, 1e-8, True)
        assert rep.true_relative_residual <= 1.05e-8
        assert abs(rep.iterations - ref.iterations) <= 2 * max(1, rep.refinements)
        assert np.abs(faces - expected).max() <= 1e-5 * np.abs(expected).max()
        # Again: the same launch over reused words gives the same bits.
        again, same = solve(hip, solver, 1e-8, False)
        assert again.iterations == rep.iterations
        assert np.array_equal(same, faces)


def test_persistent_resumes_and_stops_at_its_budget():
    # A long thin channel: more iterations than one launch takes (4096), each
    # solve resumed from the last launch's state; then a budget it cannot meet.
    grid = msa.Grid(9000, 16, 1, 1.0, 1.0, 1.0)
    rng = np.random.default_rng(5)
    mobility = rng.uniform(0.2, 5.0, (9000, 16)).astype(np.float32)
    with msa.HipBackend(0) as hip:
        hip.flow_prepare(grid, mobility, 0)
        rep, faces = solve(hip, msa.SOLVER_JACOBI_FP64, 1e-8, False)
        ref, expected = solve(hip, msa.SOLVER_JACOBI_FP64, 1e-8, True)
        assert rep.iterations > 4096
        # Over so many iterations the sums' order moves the count by its own
        # rounding: within a thousandth.
        assert abs(rep.iterations - ref.iterations) <= max(2, ref.iterations // 1000)
        assert np.abs(faces - expected).max() <= 1e-4 * np.abs(expected).max()
        for budget in (1, 7, 4096, 4100):
            for profile in (False, True):
                with pytest.raises(msa.NotConverged):
                    solve(hip, msa.SOLVER_JACOBI_FP64, 1e-8, profile, budget)
        rep2, faces2 = solve(hip, msa.SOLVER_JACOBI_FP64, 1e-8, False)
        assert rep2.iterations == rep.iterations and np.array_equal(faces2, faces)
