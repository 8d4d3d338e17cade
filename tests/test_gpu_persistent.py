"""Jacobi-PCG as one persistent launch (small and medium systems) against the
same iteration as two launches each: the pressure's, which a profiled solve
takes by launches, and the resolved flow's momentum solves, which take launches
on a context that allows no resident workgroups.

Both stop on the same test of the same recurrence and differ in the order of
their FP64 sums only, so the iteration counts agree within the reference's own
allowance of 2 (tests/conformance/flow_conformance_test.cpp:259-263). Their
fields differ by what an iteration leaves at the stated residual, bounded for
these systems by 1e-5 of the largest speed as in the other solver-form tests.
"""
import threading

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
    (520, 2017), (300, 3600),        # more sites than are taken: the same launches
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


@pytest.mark.parametrize("nx,ny", [(64, 48), (512, 256), (40, 1400)])
@pytest.mark.parametrize("solver", [msa.SOLVER_JACOBI_FP64, msa.SOLVER_MIXED])
def test_a_persistent_launch_given_up_falls_back_to_launches(nx, ny, solver):
    # A launch that ends without an iteration, as one given up does: the solve
    # starts over by launches, to their bits. Then as before.
    grid, mobility = system(nx, ny, 3)
    with msa.HipBackend(0) as hip:
        hip.flow_prepare(grid, mobility, 0)
        limits = hip.resident_limits()
        rep, faces = solve(hip, solver, 1e-8, False)
        hip.set_resident_limits(workgroups=0)
        ref, expected = solve(hip, solver, 1e-8, False)
        hip.set_resident_limits(workgroups=limits["workgroups"], iterations=0)
        got, fell_back = solve(hip, solver, 1e-8, False)
        assert got.iterations == ref.iterations
        assert np.array_equal(fell_back, expected)
        hip.set_resident_limits(iterations=limits["iterations"])
        again, same = solve(hip, solver, 1e-8, False)
        assert again.iterations == rep.iterations
        assert np.array_equal(same, faces)


@pytest.mark.parametrize("solver", [msa.SOLVER_JACOBI_FP64, msa.SOLVER_MIXED])
def test_a_device_with_less_lds_takes_launches(solver):
    # 512x256 FP64 sites: 2048 own and 2 x 256 beside them, 20.5 KB.
    grid, mobility = system(512, 256, 3)
    with msa.HipBackend(0) as hip:
        hip.flow_prepare(grid, mobility, 0)
        hip.set_resident_limits(workgroups=0)
        ref, expected = solve(hip, solver, 1e-8, False)
        hip.set_resident_limits(workgroups=256, lds_bytes=8192)
        got, faces = solve(hip, solver, 1e-8, False)
        assert got.iterations == ref.iterations
        assert np.array_equal(faces, expected)


def test_resident_limits_are_clamped_and_checked():
    with msa.HipBackend(0) as hip:
        most = hip.resident_limits()
        assert most["workgroups"] > 0 and most["iterations"] > 0
        hip.set_resident_limits(workgroups=0xffffffff, iterations=0xffffffff,
                                lds_bytes=0xffffffff, round_tag=9)
        hip.set_resident_limits(round_tag=3)
        assert hip.resident_limits() == {**most, "round_tag": 9}
        with pytest.raises(TypeError):
            hip.set_resident_limits(blocks=1)


@pytest.mark.parametrize("solver", [msa.SOLVER_JACOBI_FP64, msa.SOLVER_MIXED])
def test_meetings_start_over_before_their_number_wraps(solver):
    grid, mobility = system(131, 77, 1)
    with msa.HipBackend(0) as hip:
        hip.flow_prepare(grid, mobility, 0)
        rep, faces = solve(hip, solver, 1e-8, False)
        hip.set_resident_limits(round_tag=0xffffffff - 3 * 8192)
        for _ in range(6):
            again, same = solve(hip, solver, 1e-8, False)
            assert again.iterations == rep.iterations
            assert np.array_equal(same, faces)
        assert hip.resident_limits()["round_tag"] < 0x80000000


def test_two_contexts_solve_at_once():
    # Each context has its own words: solves of different systems in two
    # threads give what each gives alone.
    cases = [(131, 77, msa.SOLVER_JACOBI_FP64), (512, 256, msa.SOLVER_MIXED)]
    alone = []
    for nx, ny, solver in cases:
        grid, mobility = system(nx, ny, 2)
        with msa.HipBackend(0) as hip:
            hip.flow_prepare(grid, mobility, 0)
            alone.append(solve(hip, solver, 1e-8, False))
    out = [[], []]

    def work(k):
        nx, ny, solver = cases[k]
        grid, mobility = system(nx, ny, 2)
        with msa.HipBackend(0) as hip:
            hip.flow_prepare(grid, mobility, 0)
            for _ in range(8):
                out[k].append(solve(hip, solver, 1e-8, False))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for (rep, faces), results in zip(alone, out):
        assert len(results) == 8
        for again, same in results:
            assert again.iterations == rep.iterations
            assert np.array_equal(same, faces)


@pytest.mark.parametrize("nx,ny,solver,taken", [
    (500, 1792, msa.SOLVER_JACOBI_FP64, True),    # 60 KB of LDS to the byte
    (500, 1793, msa.SOLVER_JACOBI_FP64, False),
    (280, 3600, msa.SOLVER_JACOBI_FP64, False),
    (280, 3600, msa.SOLVER_MIXED, True),          # half of it
])
def test_the_lds_limit_decides(nx, ny, solver, taken):
    # Fewer sites than the most that are taken: the halo of ny sites either side
    # decides. A persistent launch numbers its meetings.
    grid, mobility = system(nx, ny, 6)
    with msa.HipBackend(0) as hip:
        hip.flow_prepare(grid, mobility, 0)
        workgroups = hip.resident_limits()["workgroups"]
        hip.set_resident_limits(workgroups=0)
        ref, expected = solve(hip, solver, 1e-8, False)
        hip.set_resident_limits(workgroups=workgroups)
        before = hip.resident_limits()["round_tag"]
        rep, faces = solve(hip, solver, 1e-8, False)
        assert (hip.resident_limits()["round_tag"] > before) == taken
    assert abs(rep.iterations - ref.iterations) <= 2 * max(1, rep.refinements)
    assert np.abs(faces - expected).max() <= 1e-5 * np.abs(expected).max()


def test_persistent_launches_of_few_iterations_go_on_to_the_same_bits():
    grid, mobility = system(131, 77, 4)
    with msa.HipBackend(0) as hip:
        hip.flow_prepare(grid, mobility, 0)
        rep, faces = solve(hip, msa.SOLVER_JACOBI_FP64, 1e-8, False)
        for iterations in (1, 37):
            hip.set_resident_limits(iterations=iterations)
            again, same = solve(hip, msa.SOLVER_JACOBI_FP64, 1e-8, False)
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


def resolved_system(dims):
    rng = np.random.default_rng(sum(dims))
    solid = (rng.random(dims) < 0.06).astype(np.uint8)
    solid[0] = solid[-1] = 0
    grid = msa.Grid(*dims, 1.0, 0.9, 1.1, solid.reshape(-1))
    return grid, (rng.random(dims) * 2.0).astype(np.float32).reshape(-1)


def resolved(hip, grid, drag, tolerance, most=50_000):
    field, rep = hip.solve_resolved_flow(grid, drag, msa.ResolvedFlowParameters(
        mean_inlet_speed=1.0, axis=0, relative_tolerance=tolerance, max_outer_iterations=4000,
        max_inner_iterations=most))
    return field.concatenated(), rep


# Launches that end without an iteration, as one given up does; that end at
# their iterations, from the first momentum solve on (3) or a later one (None:
# between the shortest and the longest).
@pytest.mark.parametrize("iterations", [0, 3, None])
@pytest.mark.parametrize("dims", [(12, 9, 7), (7, 40, 30), (40, 20, 18)])
def test_a_momentum_launch_left_undone_falls_back_to_launches(dims, iterations):
    grid, drag = resolved_system(dims)
    with msa.HipBackend(0) as hip:
        limits = hip.resident_limits()
        faces, rep = resolved(hip, grid, drag, 1e-6)
        hip.set_resident_limits(workgroups=0)
        expected, ref = resolved(hip, grid, drag, 1e-6)
        hip.set_resident_limits(workgroups=limits["workgroups"])
        mean = rep.inner_iterations // rep.outer_iterations
        hip.set_resident_limits(iterations=mean if iterations is None else iterations)
        got, again = resolved(hip, grid, drag, 1e-6)
        # Steps before the one redone were the persistent form's.
        assert abs(again.outer_iterations - ref.outer_iterations) <= 1
        if iterations is not None:
            assert again.inner_iterations == ref.inner_iterations
            assert np.array_equal(got, expected)
        else:
            assert np.abs(got - expected).max() <= 3e-5 * np.abs(expected).max()
        # The caller's own limit on the iterations is what is refused, in either
        # form, also where it is past the launch's.
        for most in (2, 5):
            with pytest.raises(msa.NotConverged, match="momentum conjugate gradient did not"):
                resolved(hip, grid, drag, 1e-6, most)
        hip.set_resident_limits(**limits)
        same, once = resolved(hip, grid, drag, 1e-6)
        assert once.inner_iterations == rep.inner_iterations
        assert np.array_equal(same, faces)


# Faces per workgroup are 512, 1024, 2048 or 4096 by the count; the halo is a
# plane of the lattice either side, here also more than a workgroup's faces.
@pytest.mark.parametrize("dims,tolerance", [
    ((5, 4, 3), 1e-6), ((1, 6, 5), 1e-6), ((12, 9, 7), 1e-6), ((20, 15, 11), 1e-6),
    ((7, 40, 30), 1e-6), ((40, 20, 18), 1e-5), ((3, 60, 61), 1e-6), ((72, 50, 49), 1e-2),
])
def test_momentum_persistent_matches_launches(dims, tolerance):
    grid, drag = resolved_system(dims)
    out = []
    with msa.HipBackend(0) as hip:
        for workgroups in (hip.resident_limits()["workgroups"], 0):
            hip.set_resident_limits(workgroups=workgroups)
            out.append(resolved(hip, grid, drag, tolerance))
    (faces, rep), (expected, ref) = out
    # The same FP64 recurrences with their sums in another order: an inner
    # solve may stop one iteration apart, an outer cycle one step.
    assert abs(rep.outer_iterations - ref.outer_iterations) <= 1
    assert abs(rep.inner_iterations - ref.inner_iterations) <= 2 + ref.inner_iterations // 100
    # 1e-6 for what the stopping test leaves at 1e-6, in proportion above it
    # (at equal counts the two differ by rounding only, 1e-7 of FP32 faces).
    bound = 1e-6 if rep.outer_iterations == ref.outer_iterations else 30 * tolerance
    assert np.abs(faces - expected).max() <= bound * np.abs(expected).max()
