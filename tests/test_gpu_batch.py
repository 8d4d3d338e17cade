"""The batched sweep on the GPU through the C ABI.

- Pressure: FP32 corrections by conjugate gradient with the multilevel cycle
  (FP64 dot products) inside FP64 refinement of each instance's FP64 pressure, to FP64 true relative residual
  1e-10, against the FP64 oracle's solve of the same instance (mo_flow_solve,
  unscaled, times the inlet pressure, to 1e-13): the device's residual equals
  the one recomputed with the oracle's operator (mo_flow_apply) to 1e-6
  relative, and face velocities agree within 1e-5 of the largest speed.
- Transport: one batched step is the single-grid FP32 step bit for bit (the
  oracle's mo_adr_step_f32 on the faces the batched step used).
- Graph: replays of a captured run, with eager work between them, equal the
  eager run bit for bit.
- Ledger: the FP64 masses it records are the masses of the levels, and the
  pressure residual each step checks is the solve's.
"""
from __future__ import annotations

import numpy as np
import pytest

import microsimulator_amd as msa
from microsimulator_amd.workloads import batch_instance
from oracle import Grid as OGrid

pytestmark = pytest.mark.gpu

SEED = 11


def small_batch():
    inst = [batch_instance(k, SEED) for k in range(7)]
    assert len({(i.nx, i.ny) for i in inst}) >= 3  # uneven sizes
    return inst


def stable_dt(hip, instances):
    worst = 0.0
    for k, inst in enumerate(instances):
        f = hip.batch_download(k)
        speed = max(float(np.abs(f["x_faces"]).max()), float(np.abs(f["y_faces"]).max()))
        phi = 0.0 if inst.phi is None else float(np.max(inst.phi))
        bound = (2.0 * inst.diffusion * (1.0 / inst.dx ** 2 + 1.0 / inst.dy ** 2)
                 + 2.0 * speed / min(inst.dx, inst.dy) + 1.0 * phi / 0.1)
        worst = max(worst, bound)
    return 0.5 / worst


def ogrid(inst):
    return OGrid(inst.nx, inst.ny, 1, inst.dx, inst.dy, inst.dz, inst.obstacles)


def test_batch_flow_matches_the_oracle(hip, oracle):
    inst = small_batch()
    hip.batch_upload(inst, relative_tolerance=1e-10, max_iterations=40000)
    it, res, fl = hip.batch_solve_flow()
    print("iterations", it.tolist(), "residuals", res.tolist(), flush=True)
    assert np.all(fl == 0)
    assert np.all(res <= 1e-10)
    for k, i in enumerate(inst):
        g = ogrid(i)
        f = hip.batch_download(k)
        # The right-hand side for inlet pressure p: p times the assembled one, in FP64.
        b = oracle.assemble(g, i.mobility, 0)["rhs"].astype(np.float64) * np.float64(np.float32(i.inlet_pressure))
        true = np.linalg.norm(b - oracle.apply(g, i.mobility, f["pressure"])) / np.linalg.norm(b)
        faces, _, _ = oracle.solve_flow(g, i.mobility, 0, 1.0, 1e-13, 400000, scale=False)
        ref = faces.astype(np.float64) * i.inlet_pressure
        got = np.concatenate([f["x_faces"], f["y_faces"]]).astype(np.float64)
        n = got.size
        err = np.abs(got - ref[:n]).max() / np.abs(ref[:n]).max()
        print(k, (i.nx, i.ny), "FP64 true residual", true, "velocity error / max speed", err,
              flush=True)
        assert true <= 1e-10
        assert true == pytest.approx(float(res[k]), rel=1e-6, abs=1e-15)
        assert err <= 1e-5
    # A second solve starts from the converged pressures.
    it2, _, _ = hip.batch_solve_flow()
    assert np.all(it2 <= 2)


def odd_instance(nx, ny, pocket):
    rng = np.random.default_rng([SEED, nx, ny])
    solid = np.zeros((nx, ny), np.uint8)
    if nx >= 16 and ny >= 16:
        solid[5:9, 2:ny // 2] = 1
    if pocket:  # fluid without an open boundary: zero rows and a vanishing pivot
        solid[nx // 2:nx // 2 + 7, 8:15] = 1
        solid[nx // 2 + 2:nx // 2 + 5, 10:13] = 0
    return msa.BatchInstance(nx=nx, ny=ny, mobility=rng.uniform(0.2, 2.0, nx * ny).astype(np.float32),
                             obstacles=solid.reshape(-1), inlet_pressure=1.3, dx=1.5, dy=0.75)


@pytest.mark.parametrize("sizes", [
    [(3, 3), (8, 8), (2, 31)],            # one level: the dense inverse alone
    [(13, 5), (65, 3), (3, 65), (9, 8)],  # one coarsening, odd remainders
    [(33, 31), (129, 17), (64, 64), (37, 111)],
    [(91, 91), (3, 3)],                          # over the whole chip: two tiled levels
    [(701, 300), (5, 7), (300, 47)],             # four, beside a single-level instance
])
@pytest.mark.parametrize("pocket", [False, True])
def test_batch_system_at_odd_sizes(hip, oracle, sizes, pocket):
    """The device's setup and cycle at level edges: every instance converges to
    1e-10 of the oracle's own right-hand side and operator (FP64), in no more
    iterations than a multilevel cycle needs: plain aggregation loses a fixed
    factor per level, some 13 to 18 iterations of the ten digits asked for, so
    30 per level (Jacobi alone takes several times the longer side; a wrong
    coarse operator or inverse costs hundreds or fails)."""
    inst = [odd_instance(nx, ny, pocket and nx >= 24 and ny >= 17) for nx, ny in sizes]
    hip.batch_upload(inst, relative_tolerance=1e-10, max_iterations=4000)
    it, res, fl = hip.batch_solve_flow()
    print(sizes, "iterations", it.tolist(), "residuals", res.tolist(), flush=True)
    assert np.all(fl == 0)
    for k, i in enumerate(inst):
        g = ogrid(i)
        b = oracle.assemble(g, i.mobility, 0)["rhs"].astype(np.float64) * np.float64(np.float32(i.inlet_pressure))
        true = np.linalg.norm(b - oracle.apply(g, i.mobility, hip.batch_download(k)["pressure"])) / np.linalg.norm(b)
        assert true <= 1e-10
        levels, nx, ny = 1, i.nx, i.ny
        while nx * ny > 64:
            levels, nx, ny = levels + 1, (nx + 1) // 2, (ny + 1) // 2
        assert it[k] <= 30 * levels


def test_batch_step_is_the_single_grid_step(hip, oracle):
    inst = small_batch()
    rng = np.random.default_rng(4)
    for i in inst:
        i.levels = rng.uniform(0.0, 1.0, i.sites).astype(np.float32) * (i.obstacles.reshape(-1) == 0)
    hip.batch_upload(inst, relative_tolerance=1e-8, max_iterations=40000)
    hip.batch_solve_flow()
    dt = stable_dt(hip, inst)
    hip.batch_run(dt, 1, graph=False)
    for k, i in enumerate(inst):
        f = hip.batch_download(k)
        bv = np.zeros(6, np.float32)
        bv[0] = i.reservoir
        zf = np.zeros(i.sites * 2, np.float32)
        ref = oracle.adr_step_f32(ogrid(i), i.levels, dt, diffusion=[i.diffusion],
                                  boundary_values=bv,
                                  faces=np.concatenate([f["x_faces"], f["y_faces"], zf]),
                                  phi=i.phi, vmax=1.0, monod_k=0.1)
        mismatch = int(np.count_nonzero(f["levels"] != ref))
        print(k, (i.nx, i.ny), "mismatching sites", mismatch, flush=True)
        assert mismatch == 0


def test_graph_replays_equal_the_eager_run(hip):
    inst = small_batch()
    hip.batch_upload(inst, relative_tolerance=1e-8, max_iterations=40000)
    hip.batch_solve_flow()
    dt = stable_dt(hip, inst)
    eager_led, _ = hip.batch_run(dt, 6, graph=False)
    eager_led2, _ = hip.batch_run(dt, 6, graph=False)
    eager = [hip.batch_download(k)["levels"] for k in range(len(inst))]

    hip.batch_upload(inst, relative_tolerance=1e-8, max_iterations=40000)
    hip.batch_solve_flow()
    led1, _ = hip.batch_run(dt, 6, graph=True)
    mid = [hip.batch_download(k)["levels"] for k in range(len(inst))]  # eager work between
    led2, _ = hip.batch_run(dt, 6, graph=True)                         # the same graph again
    final = [hip.batch_download(k)["levels"] for k in range(len(inst))]
    np.testing.assert_array_equal(led1, eager_led)
    np.testing.assert_array_equal(led2, eager_led2)
    for a, b in zip(final, eager):
        np.testing.assert_array_equal(a, b)
    assert any(np.any(a != b) for a, b in zip(mid, final))


def test_ledger_masses_are_the_levels(hip):
    inst = small_batch()
    hip.batch_upload(inst, relative_tolerance=1e-8, max_iterations=40000)
    hip.batch_solve_flow()
    dt = stable_dt(hip, inst)
    led, _ = hip.batch_run(dt, 5, graph=True)
    assert np.all(hip.batch_flags() == 0)
    assert np.all(led[:, :, 3] <= 1e-8)  # the pressure each step checked
    # Mass after one step is mass before the next, bit for bit.
    np.testing.assert_array_equal(led[1:, :, 0], led[:-1, :, 1])
    for k, i in enumerate(inst):
        lv = hip.batch_download(k)["levels"].astype(np.float64)
        mass = lv[i.obstacles.reshape(-1) == 0].sum() * i.dx * i.dy * i.dz
        assert led[-1, k, 1] == pytest.approx(mass, rel=1e-12)
        assert led[0, k, 0] == 0.0  # started empty
        assert led[-1, k, 1] > 0.0  # the reservoir feeds it


def test_autotune_picks_one_of_the_shapes(hip):
    inst = small_batch()
    hip.batch_upload(inst, relative_tolerance=1e-8, max_iterations=40000)
    hip.batch_solve_flow()
    dt = stable_dt(hip, inst)
    eager, _ = hip.batch_run(dt, 3, graph=False)
    ref = [hip.batch_download(k)["levels"] for k in range(len(inst))]
    hip.batch_upload(inst, relative_tolerance=1e-8, max_iterations=40000)
    hip.batch_solve_flow()
    shape, secs = hip.batch_autotune(dt, steps=2)
    print("shape", hip.batch_shapes()[shape], "per-step seconds", secs.tolist(), flush=True)
    assert 0 <= shape < len(hip.batch_shapes())
    assert np.all(secs > 0.0)
    assert secs[shape] == secs.min()
    hip.batch_run(dt, 3, graph=True)
    for k, a in enumerate(ref):  # any shape computes every site the same way
        np.testing.assert_array_equal(hip.batch_download(k)["levels"], a)


def test_batch_rejects_bad_instances(hip):
    inst = small_batch()[:2]
    inst[1].mobility = inst[1].mobility.copy()
    inst[1].mobility[3] = -1.0
    with pytest.raises(msa.InvalidArgument):
        hip.batch_upload(inst)
    with pytest.raises(msa.InvalidArgument):
        hip.batch_upload(inst[:1], relative_tolerance=0.0)


@pytest.mark.parametrize("shape", [(16, 12), (128, 96)])  # one workgroup; the whole chip
def test_a_solve_without_a_finite_residual_is_flagged(hip, shape):
    """A conductance past the largest float leaves no finite residual: the
    instance is flagged as broken down, and its neighbour solves as ever.
    (The one-workgroup form ended without a flag.)"""
    nx, ny = shape
    mobility = np.ones((nx, ny), np.float32)
    wild = mobility.copy()
    wild[nx // 2:] = 3.0e38

    def instance(m):
        return msa.BatchInstance(nx=nx, ny=ny, mobility=m, inlet_pressure=1.0, reservoir=1.0,
                                 diffusion=1.0, dx=1.0, dy=1.0, dz=10.0)

    hip.batch_upload([instance(wild), instance(mobility)], relative_tolerance=1e-8,
                     max_iterations=2000)
    it, res, flags = hip.batch_solve_flow()
    assert flags[0] & 1
    assert flags[1] == 0 and res[1] <= 1e-8 and it[1] > 0
