"""The work a user of this backend has it do, as timed cases.

Every case runs through the public Python entry points of
``microsimulator_amd.HipBackend``. ``listed()`` gives the fixed cases,
``draw()`` more of the same ranges, ``prepare()`` what a program holds before
the call (geometry, the prepared system or the uploaded state), ``run()`` one
pass with its whole outputs, ``exact()`` the same outputs in FP64 by plain
torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import microsimulator_amd as msa
from microsimulator_amd import learned, workloads

SPEED = 100.0  # mean inlet speed of every flow, lengths per second
VMAX, HALF = 1.0, 0.1  # Monod uptake
DIFFUSION = (100.0, 500.0, 1000.0)
SOLVERS = {"fp64": msa.SOLVER_JACOBI_FP64, "mixed": msa.SOLVER_MIXED,
           "learned": msa.SOLVER_LEARNED, "multigrid": msa.SOLVER_MULTIGRID}
BOUNDARY = (msa.FIXED, msa.FIXED, msa.NO_FLUX, msa.NO_FLUX, msa.NO_FLUX, msa.NO_FLUX)


def listed():
    return [
        # One ComputeBackend step of a small device, as a simulation loop that
        # keeps its levels on the host calls it: latency and launches.
        dict(name="step_64x48", kind="step", geometry="trap", nx=64, ny=48, signals=1,
             scheme="upwind"),
        # The reference's own call on the channel-and-trap device: validation,
        # upload, FP64 Jacobi-PCG, field back on the host.
        dict(name="call_fp64_256x128", kind="call", geometry="trap", nx=256, ny=128,
             solver="fp64", tolerance=1e-10),
        # A medium pillar array by FP32 Jacobi-PCG with FP64 refinement.
        dict(name="solve_mixed_1024x512", kind="solve", geometry="pillars", nx=1024, ny=512,
             solver="mixed", tolerance=1e-8),
        # The trap device at the training size of the learned smoother.
        dict(name="solve_learned_512x256", kind="solve", geometry="trap", nx=512, ny=256,
             solver="learned", tolerance=1e-8),
        # A ragged pillar array by the multilevel form.
        dict(name="solve_multigrid_3001x1777", kind="solve", geometry="pillars", nx=3001,
             ny=1777, solver="multigrid", tolerance=1e-8),
        # The large pillar array by the headline form.
        dict(name="solve_learned_4096x2048", kind="solve", geometry="pillars", nx=4096, ny=2048,
             solver="learned", tolerance=1e-8),
        # Long FP64 transport with its mass ledger on the large array, the
        # levels fetched every few hundred steps.
        dict(name="adr_fp64_4096x2048", kind="transport", geometry="pillars", nx=4096, ny=2048,
             signals=3, precision=64, scheme="upwind", integration="euler", steps=400),
        # FP32 van Leer transport on a ragged device.
        dict(name="adr_vl_1531x769", kind="transport", geometry="pillars", nx=1531, ny=769,
             signals=2, precision=32, scheme="van_leer", integration="euler", steps=200),
        # Crank-Nicolson transport at four times the explicit bound.
        dict(name="adr_cn_2048x1024", kind="transport", geometry="pillars", nx=2048, ny=1024,
             signals=3, precision=32, scheme="upwind", integration="crank_nicolson", steps=20),
        # A large colony exchanging three solutes with the large array.
        dict(name="coupled_4096x2048", kind="coupled", geometry="pillars", nx=4096, ny=2048,
             cells=1 << 20, steps=100),
        # A design sweep from upload to results: pressure, 50 steps, every
        # instance fetched.
        dict(name="sweep_256", kind="sweep", instances=256, steps=50, tolerance=1e-8),
        # A three-dimensional channel by the resolved solver.
        dict(name="resolved_64x32x16", kind="resolved", nx=64, ny=32, nz=16, tolerance=1e-6),
    ]


def _between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("step", "call", "solve", "solve", "transport", "transport", "coupled",
                       "sweep", "resolved"))
    geometry = rng.choice(("pillars", "trap"))
    if kind == "step":
        return dict(kind=kind, geometry=geometry, nx=_between(rng, 64, 768),
                    ny=_between(rng, 48, 512), signals=rng.randint(1, 3),
                    scheme=rng.choice(("upwind", "van_leer")))
    if kind == "call":
        return dict(kind=kind, geometry=geometry, nx=_between(rng, 64, 512),
                    ny=_between(rng, 48, 256), solver="fp64",
                    tolerance=rng.choice((1e-8, 1e-10)))
    if kind == "solve":
        solver = rng.choice(("mixed", "learned", "multigrid"))
        most = 2 if solver == "mixed" else 8
        return dict(kind=kind, geometry=geometry, nx=_between(rng, 256, 512 * most),
                    ny=_between(rng, 128, 256 * most), solver=solver, tolerance=1e-8)
    if kind == "transport":
        precision, scheme, integration, steps = rng.choice(
            ((64, "upwind", "euler", 400), (32, "upwind", "euler", 400),
             (32, "van_leer", "euler", 200), (32, "upwind", "crank_nicolson", 20)))
        most = 4 if integration != "euler" else 8
        return dict(kind=kind, geometry="pillars", nx=_between(rng, 256, 512 * most),
                    ny=_between(rng, 128, 256 * most), signals=rng.randint(1, 3),
                    precision=precision, scheme=scheme, integration=integration, steps=steps)
    if kind == "coupled":
        nx, ny = _between(rng, 256, 4096), _between(rng, 128, 2048)
        return dict(kind=kind, geometry="pillars", nx=nx, ny=ny, cells=nx * ny // 8, steps=100)
    if kind == "sweep":
        return dict(kind=kind, instances=_between(rng, 24, 256), steps=rng.randint(20, 50),
                    tolerance=1e-8)
    return dict(kind=kind, nx=_between(rng, 24, 64), ny=_between(rng, 16, 32),
                nz=_between(rng, 8, 16), tolerance=1e-6)


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _pillars(nx, ny, seed):
    """A channel of seeded circular pillars on a jittered lattice (about one
    per 2000 sites, radii U[8, 20], smaller on narrow channels), biomass from
    Gaussian blobs, a depth of 8 to 12 per site."""
    rng = np.random.default_rng(seed)
    scale = min(1.0, ny / 512.0)
    pitch = max(12.0, 46.0 * scale)
    kx, ky = max(1, int((nx - 2 * pitch) // pitch)), max(1, int(ny // pitch))
    radius = rng.uniform(8.0 / 46.0, 20.0 / 46.0, (kx, ky)) * pitch
    room = np.maximum(0.0, 0.5 * pitch - radius - 1.0)
    cx = pitch * (1.5 + np.arange(kx))[:, None] + rng.uniform(-1, 1, (kx, ky)) * room
    cy = pitch * (0.5 + np.arange(ky))[None, :] + rng.uniform(-1, 1, (kx, ky)) * room
    dev = _device()
    x = torch.arange(nx, device=dev, dtype=torch.float64) + 0.5
    y = torch.arange(ny, device=dev, dtype=torch.float64) + 0.5
    ix = torch.clamp((x / pitch - 1.0).floor().long(), 0, kx - 1)[:, None]
    iy = torch.clamp((y / pitch).floor().long(), 0, ky - 1)[None, :]
    tx, ty, tr = (torch.as_tensor(a, device=dev) for a in (cx, cy, radius))
    solid = (x[:, None] - tx[ix, iy]) ** 2 + (y[None, :] - ty[ix, iy]) ** 2 <= tr[ix, iy] ** 2
    blobs = max(2, nx * ny // 16777)
    bx, by = (torch.as_tensor(rng.uniform(0, n, blobs), device=dev) for n in (nx, ny))
    sigma = torch.as_tensor(rng.uniform(10.0, 30.0, blobs) * scale, device=dev)
    peak = torch.as_tensor(rng.uniform(0.3, 0.7, blobs), device=dev)
    gx = torch.exp(-((x[:, None] - bx) ** 2) / (2 * sigma**2))
    gy = torch.exp(-((y[:, None] - by) ** 2) / (2 * sigma**2))
    phi = torch.clamp((gx * peak) @ gy.T, max=0.7)
    depth = torch.as_tensor(rng.uniform(8.0, 12.0, (nx, ny)), device=dev)
    k = depth * depth / 12.0
    drag = workloads.DRAG_COEFFICIENT * phi * phi / (1.0 - phi) ** 3
    mobility = torch.where(solid, 0.0, depth / 10.0 * k / (1.0 + k * drag)).float()
    phi = torch.where(solid, 0.0, phi).float()
    return workloads.Workload("pillars", nx, ny, 1.0, 1.0, 10.0,
                              solid.to(torch.uint8).cpu().numpy(), mobility.cpu().numpy(),
                              phi.cpu().numpy())


def _geometry(case, seed):
    if case["geometry"] == "pillars":
        return _pillars(case["nx"], case["ny"], seed)
    return workloads.channel_trap(case["nx"], case["ny"], seed=seed)


def _grid(w):
    return msa.Grid(w.nx, w.ny, 1, w.dx, w.dy, w.dz, w.obstacles, BOUNDARY)


def _levels(w, signals, seed, dtype):
    """Smooth seeded levels in [0.1, 0.9], zero at solids."""
    rng = np.random.default_rng([seed, 1])
    x, y = np.arange(w.nx) / w.nx, np.arange(w.ny) / w.ny
    out = np.empty((signals, w.nx, w.ny), dtype)
    for s in range(signals):
        a, b, c, d = rng.uniform(1.0, 4.0, 4)
        out[s] = 0.5 + 0.4 * np.sin(2 * np.pi * (a * x + b))[:, None] * np.cos(
            2 * np.pi * (c * y + d))[None, :]
    out[:, w.obstacles != 0] = 0.0
    return out


def _reservoirs(signals):
    values = np.zeros(6 * signals, np.float32)
    values[0::6] = 1.0
    return values


def _outflow(field, nx, ny):
    xf, yf = field.x_faces.reshape(nx + 1, ny), field.y_faces.reshape(nx, ny + 1)
    return float((np.maximum(xf[1:], 0) - np.minimum(xf[:-1], 0)
                  + np.maximum(yf[:, 1:], 0) - np.minimum(yf[:, :-1], 0)).max())


def _step(share, rate):
    """share / rate to three digits: a step does not depend on the last bits
    of the speeds its bound is taken from."""
    dt = share / rate
    digit = 10.0 ** math.floor(math.log10(dt)) / 100
    return math.floor(dt / digit) * digit


def _bound_rate(w, outflow, signals, scheme):
    """One over the largest step the explicit stability bound allows."""
    courant = 2.0 * outflow if scheme == "van_leer" else outflow
    return 4.0 * max(DIFFUSION[:signals]) + courant + VMAX * float(w.phi.max()) / HALF


def _flow_parameters(case):
    return msa.DepthAveragedFlowParameters(
        mean_inlet_speed=SPEED, axis=0, relative_tolerance=case["tolerance"],
        max_iterations=200_000, solver=SOLVERS[case["solver"]])


def _solved(hip, w):
    """A converged flow on the device: its field and the system behind it."""
    hip.flow_prepare(_grid(w), w.mobility, 0)
    hip.flow_solve(msa.DepthAveragedFlowParameters(
        mean_inlet_speed=SPEED, axis=0, relative_tolerance=1e-8, max_iterations=2000,
        solver=msa.SOLVER_MULTIGRID))
    return hip.flow_download()[1]


def _spec(case, w, velocity=None):
    S = case["signals"]
    return msa.SignalGridSpec(
        _grid(w), np.asarray(DIFFUSION[:S], np.float32), _reservoirs(S), velocity=velocity,
        phi=w.phi, monod_vmax=[VMAX] * S, monod_k=[HALF] * S,
        advection_scheme=msa.VAN_LEER if case["scheme"] == "van_leer" else msa.UPWIND,
        integration=msa.CRANK_NICOLSON if case.get("integration") == "crank_nicolson"
        else msa.FORWARD_EULER)


def _instances(case, seed):
    """A sweep's devices: the four batch sizes in an order of their own, each
    a seeded trap or pillar device with its own drive and solute."""
    sizes = np.random.default_rng(3).permutation(
        [workloads.BATCH_SIZES[k % 4] for k in range(case["instances"])])
    rng = np.random.default_rng(seed)
    out = []
    for k, (nx, ny) in enumerate(sizes.tolist()):
        gseed = int(rng.integers(1 << 30))
        if k % 2 == 0:
            w = workloads.channel_trap(nx, ny, seed=gseed)
        else:
            area = nx * ny / (1024 * 512)
            low = max(3, round(8 * ny / 512))
            w = workloads.pillar_array(
                nx, ny, seed=gseed, pillars=max(2, round(300 * area)),
                radius=(low, max(low + 1, round(15 * ny / 512))), blobs=max(2, round(40 * area)))
        out.append(msa.BatchInstance(
            nx=nx, ny=ny, mobility=w.mobility, obstacles=w.obstacles, phi=w.phi,
            inlet_pressure=float(rng.uniform(0.5, 2.0)), reservoir=1.0,
            diffusion=float(rng.uniform(100.0, 1000.0)), dx=w.dx, dy=w.dy, dz=w.dz))
    return out


def _resolved_inputs(case, seed):
    rng = np.random.default_rng(seed)
    shape = (case["nx"], case["ny"], case["nz"])
    solid = (rng.random(shape) < 0.08).astype(np.uint8)
    solid[0] = solid[-1] = 0
    drag = (rng.random(shape) * 2.0).astype(np.float32)
    return solid, drag


def prepare(case, seed):
    kind = case["kind"]
    hip = msa.HipBackend(0)
    state = dict(kind=kind, hip=hip)
    if kind in ("step", "call", "solve", "transport", "coupled"):
        w = _geometry(case, seed)
        grid = _grid(w)
    if kind == "step":
        field = _solved(hip, w)
        state.update(spec=_spec(case, w, field),
                     levels=_levels(w, case["signals"], seed, np.float32).reshape(-1),
                     dt=_step(0.9, _bound_rate(w, _outflow(field, w.nx, w.ny), case["signals"],
                                               case["scheme"])))
    elif kind == "call":
        state.update(grid=grid, mobility=w.mobility, parameters=_flow_parameters(case))
    elif kind == "solve":
        if case["solver"] == "learned":
            hip.learned_set_weights(learned.load_weights())
        hip.flow_prepare(grid, w.mobility, 0)
        state.update(parameters=_flow_parameters(case))
    elif kind == "transport":
        rate = _bound_rate(w, _outflow(_solved(hip, w), w.nx, w.ny), case["signals"],
                           case["scheme"])
        dtype = np.float64 if case["precision"] == 64 else np.float32
        hip.adr_upload(_spec(case, w), _levels(w, case["signals"], seed, dtype),
                       precision=case["precision"], use_flow_field=True)
        state.update(steps=case["steps"], ledger=case["precision"] == 64,
                     dt=_step(4.0 if case["integration"] == "crank_nicolson" else 0.9, rate))
    elif kind == "coupled":
        field = _solved(hip, w)
        cells, previous = workloads.colony(w, case["cells"], seed=seed)
        spec = msa.SignalGridSpec(grid, np.asarray(DIFFUSION, np.float32), _reservoirs(3),
                                  velocity=field)
        hip.coupled_upload(spec, _levels(w, 3, seed, np.float32), cells,
                           np.ones(2 * case["cells"], np.float32), workloads.quorum_plan())
        state.update(steps=case["steps"], previous=previous,
                     dt=_step(0.9, 4.0 * max(DIFFUSION) + _outflow(field, w.nx, w.ny)))
    elif kind == "sweep":
        instances = _instances(case, seed)
        hip.batch_upload(instances, relative_tolerance=case["tolerance"], max_iterations=60000)
        hip.batch_solve_flow()
        worst = 0.0
        for k, inst in enumerate(instances):
            f = hip.batch_download(k)
            field = msa.VelocityField(f["x_faces"], f["y_faces"], None)
            worst = max(worst, 4.0 * inst.diffusion + _outflow(field, inst.nx, inst.ny)
                        + VMAX * float(inst.phi.max()) / HALF)
        state.update(instances=instances, steps=case["steps"], tolerance=case["tolerance"],
                     dt=_step(0.9, worst))
    else:
        solid, drag = _resolved_inputs(case, seed)
        state.update(grid=msa.Grid(case["nx"], case["ny"], case["nz"], 1.0, 1.0, 1.0,
                                   solid.reshape(-1), BOUNDARY), drag=drag.reshape(-1),
                     parameters=msa.ResolvedFlowParameters(
                         mean_inlet_speed=1.0, axis=0, relative_tolerance=case["tolerance"],
                         max_outer_iterations=8000))
    return state


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
def _faces(field):
    return dict(x_faces=field.x_faces, y_faces=field.y_faces, z_faces=field.z_faces)


def run(state):
    kind, hip = state["kind"], state["hip"]
    if kind == "step":
        levels, _ = hip.advance_signal_grid(state["spec"], state["levels"], state["dt"])
        return dict(levels=levels)
    if kind == "call":
        result = hip.solve_depth_averaged_flow(state["grid"], state["mobility"],
                                               state["parameters"])
        return _faces(result.field)
    if kind == "solve":
        hip.flow_solve(state["parameters"])
        # The field, as the one-call form returns it (a pressure has no meaning
        # inside the solids, where each form leaves its own values).
        return _faces(hip.flow_download()[1])
    if kind == "transport":
        ledger = hip.adr_run(state["dt"], state["steps"], ledger=state["ledger"])
        out = dict(levels=hip.adr_download())
        if ledger is not None:
            out["ledger"] = ledger
        return out
    if kind == "coupled":
        hip.coupled_run(state["dt"], state["steps"], state["previous"])
        levels, species = hip.coupled_download()
        return dict(levels=levels, species=species)
    if kind == "sweep":
        hip.batch_upload(state["instances"], relative_tolerance=state["tolerance"],
                         max_iterations=60000)
        hip.batch_solve_flow()
        ledger, _ = hip.batch_run(state["dt"], state["steps"])
        got = [hip.batch_download(k) for k in range(len(state["instances"]))]
        out = {name: np.concatenate([g[name] for g in got])
               for name in ("x_faces", "y_faces", "levels")}
        out["masses"] = ledger[:, :, :3]
        return out
    field, _ = hip.solve_resolved_flow(state["grid"], state["drag"], state["parameters"])
    return _faces(field)


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    """Inputs read once and outputs written once, and the operations of one
    application of what is iterated: iteration counts are a method's own."""
    kind = case["kind"]
    if kind == "sweep":
        n = case["instances"] * (64 * 64 + 128 * 96 + 256 * 128 + 512 * 256) // 4
        return dict(bytes=n * (9 + 4 + 12 + case["steps"] * 12), flops=n * case["steps"] * 60)
    n = case["nx"] * case["ny"] * case.get("nz", 1)
    if kind == "step":
        S = case["signals"]
        return dict(bytes=n * (13 + 8 * S), flops=n * S * 40)
    if kind in ("call", "solve"):
        # Mobility and mask in, faces out.
        return dict(bytes=n * (5 + 12), flops=n * 20)
    if kind == "transport":
        S, size = case["signals"], case["precision"] // 8
        return dict(bytes=n * case["steps"] * (13 + 2 * S * size),
                    flops=n * case["steps"] * S * 40)
    if kind == "coupled":
        per_cell = 32 + 16 + 12
        return dict(bytes=case["steps"] * (n * (9 + 24) + case["cells"] * per_cell),
                    flops=case["steps"] * (n * 3 * 30 + case["cells"] * 100))
    return dict(bytes=n * (5 + 12), flops=n * 100)


def tolerance(case):
    """About four times the largest error against exact() seen over the listed
    and a few drawn cases (the resolved flow: against a solve to a seventh of
    its tolerance). What an iteration leaves at its stopping test outweighs
    rounding in the flows and the implicit transport."""
    kind = case["kind"]
    if kind == "step":
        return dict(rel=2e-7, max=2e-6)
    if kind in ("call", "solve"):
        if case["solver"] in ("fp64", "mixed"):
            if case["tolerance"] < 1e-9:
                return dict(rel=1e-5, max=2e-4)
            return dict(rel=1e-3, max=2e-2)
        return dict(rel=1e-5, max=5e-4)
    if kind == "transport":
        if case["integration"] == "crank_nicolson":
            return dict(rel=2e-5, max=5e-4)
        return dict(rel=3e-6, max=3e-5)
    if kind == "coupled":
        return dict(rel=3e-6, max=5e-5)
    if kind == "sweep":
        return dict(rel=3e-6, max=2e-4)
    return dict(rel=3e-4, max=1e-3)


# --------------------------------------------------------------------------
# The same outputs in 64 bits, by plain torch
# --------------------------------------------------------------------------
class _Pressure:
    """The five-point pressure system of B equal grids, solved by conjugate
    gradient under a V(2,2) aggregation cycle, all in FP64."""

    def __init__(self, cond, dx):
        self.cond, self.dx = cond, dx
        s = 1.0 / dx**2
        self.hx, self.hy = (self._harmonic(cond[:, 1:], cond[:, :-1]),
                            self._harmonic(cond[:, :, 1:], cond[:, :, :-1]))
        self.bc = torch.zeros_like(cond)
        self.bc[:, 0] += 2.0 * cond[:, 0] * s
        self.bc[:, -1] += 2.0 * cond[:, -1] * s
        self.rhs = torch.zeros_like(cond)
        self.rhs[:, 0] = 2.0 * cond[:, 0] * s
        self.levels = [self._level(self.hx * s, self.hy * s, self.bc)]
        while self.levels[-1][2][0].numel() > 64:
            self.levels.append(self._coarse(*self.levels[-1][:3]))
        wx, wy, bc, d = self.levels[-1]
        n = bc[0].numel()
        eye = torch.eye(n, dtype=cond.dtype, device=cond.device)
        cols = [self._apply(self.levels[-1], eye[k].reshape(bc.shape[1:]).expand_as(bc)
                            ).reshape(len(bc), n) for k in range(n)]
        dense = torch.stack(cols, 2)
        # Cells without a path to a held face leave the dense system singular.
        dense = dense + torch.diag_embed(torch.where(d > 0, 1e-12 * d, 1.0).reshape(len(bc), n))
        self.inverse = torch.linalg.inv(dense)

    @staticmethod
    def _harmonic(a, b):
        return torch.where(a + b > 0, 2.0 * a * b / (a + b).clamp(min=1e-300), 0.0)

    @staticmethod
    def _level(wx, wy, bc):
        d = bc.clone()
        d[:, 1:] += wx
        d[:, :-1] += wx
        d[:, :, 1:] += wy
        d[:, :, :-1] += wy
        return wx, wy, bc, d

    @staticmethod
    def _pool(a):
        a = torch.nn.functional.pad(a, (0, a.shape[2] % 2, 0, a.shape[1] % 2))
        return a[:, ::2, ::2] + a[:, 1::2, ::2] + a[:, ::2, 1::2] + a[:, 1::2, 1::2]

    @classmethod
    def _coarse(cls, wx, wy, bc):
        x = torch.nn.functional.pad(wx[:, 1::2], (0, wx.shape[2] % 2))
        y = torch.nn.functional.pad(wy[:, :, 1::2], (0, 0, 0, wy.shape[1] % 2))
        return cls._level(x[:, :, ::2] + x[:, :, 1::2], y[:, ::2] + y[:, 1::2], cls._pool(bc))

    @staticmethod
    def _apply(level, v):
        wx, wy, bc, _ = level
        out = bc * v
        g = wx * (v[:, 1:] - v[:, :-1])
        out[:, 1:] += g
        out[:, :-1] -= g
        g = wy * (v[:, :, 1:] - v[:, :, :-1])
        out[:, :, 1:] += g
        out[:, :, :-1] -= g
        return out

    def _cycle(self, r, k=0):
        if k + 1 == len(self.levels):
            return (self.inverse @ r.reshape(len(r), -1, 1)).reshape(r.shape)
        level = self.levels[k]
        smooth = torch.where(level[3] > 0, 0.8 / level[3].clamp(min=1e-300), 0.0)
        x = smooth * r
        x = x + smooth * (r - self._apply(level, x))
        e = self._cycle(self._pool(r - self._apply(level, x)), k + 1)
        e = e.repeat_interleave(2, 1)[:, : r.shape[1]].repeat_interleave(2, 2)[:, :, : r.shape[2]]
        x = x + 1.8 * e
        for _ in range(2):
            x = x + smooth * (r - self._apply(level, x))
        return x

    def solve(self, scale=None):
        """The pressure for the inlet held at `scale` (one per grid)."""
        rhs = self.rhs if scale is None else self.rhs * scale[:, None, None]
        x, r = torch.zeros_like(rhs), rhs.clone()
        norm = (rhs * rhs).sum((1, 2))
        p, rz = None, None
        for k in range(400):
            z = self._cycle(r)
            new = (r * z).sum((1, 2))
            p = z if p is None else z + (new / rz.clamp(min=1e-300))[:, None, None] * p
            rz = new
            q = self._apply(self.levels[0], p)
            alpha = (rz / (p * q).sum((1, 2)).clamp(min=1e-300))[:, None, None]
            x += alpha * p
            r -= alpha * q
            if bool(((r * r).sum((1, 2)) <= 1e-26 * norm).all()):
                break
        return x

    def faces(self, p, solid, dz, inlet=None):
        """x and y face velocities of the pressure p."""
        dx, c = self.dx, self.cond
        held = 1.0 if inlet is None else inlet[:, None]
        x = torch.cat([(2.0 * c[:, 0] / dx * (held - p[:, 0]))[:, None],
                       -self.hx * (p[:, 1:] - p[:, :-1]) / dx,
                       (2.0 * c[:, -1] / dx * p[:, -1])[:, None]], 1)
        y = torch.nn.functional.pad(-self.hy * (p[:, :, 1:] - p[:, :, :-1]) / dx, (1, 1))
        return x / dz, y / dz


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), device=_device()).to(dtype)


def _exact_flow(w):
    """Pressure, and the faces scaled to the mean inlet speed."""
    solid = _t(w.obstacles, torch.bool)
    cond = torch.where(solid, 0.0, float(w.dz) * _t(w.mobility))[None]
    system = _Pressure(cond, float(w.dx))
    p = system.solve()
    x, y = system.faces(p, solid, float(w.dz))
    open_inlet = ~solid[0] & (cond[0, 0] > 0)
    factor = SPEED / (x[0, 0][open_inlet].mean())
    return p[0], x[0] * factor, y[0] * factor


class _Site:
    """The transport rate of [..., nx, ny] levels: fixed reservoirs at the x
    ends, closed y ends and solids."""

    def __init__(self, solid, xf, yf, dx, limited=False):
        self.fluid = ~solid
        f = self.fluid
        pad = torch.nn.functional.pad
        self.open_x = torch.cat([f[..., :1, :], f[..., 1:, :] & f[..., :-1, :], f[..., -1:, :]], -2)
        self.open_y = pad(f[..., 1:] & f[..., :-1], (1, 1), value=False)
        self.ux = torch.where(self.open_x, xf, 0.0)
        self.uy = torch.where(self.open_y, yf, 0.0)
        self.dx, self.limited = dx, limited

    def rate(self, c, diffusion, low, high):
        """`low`, `high`: reservoir levels beyond the x ends, and
        `diffusion`, broadcast against c[..., :1, :]."""
        pad = torch.nn.functional.pad
        lo, hi = low.expand_as(c[..., :1, :]), high.expand_as(c[..., :1, :])
        ext = torch.cat([lo, c, hi], -2)
        flux = torch.where(self.ux >= 0, self.ux * ext[..., :-1, :], self.ux * ext[..., 1:, :])
        flux = flux - torch.where(
            self.open_x, diffusion * (ext[..., 1:, :] - ext[..., :-1, :]), 0.0) / self.dx
        if self.limited:
            flux = flux + self._limited(c, self.ux, self.fluid, -2)
        out = -(flux[..., 1:, :] - flux[..., :-1, :]) / self.dx
        ext = pad(c, (1, 1))
        flux = torch.where(self.uy >= 0, self.uy * ext[..., :-1], self.uy * ext[..., 1:])
        flux = flux - torch.where(
            self.open_y, diffusion * (ext[..., 1:] - ext[..., :-1]), 0.0) / self.dx
        if self.limited:
            flux = flux + self._limited(c, self.uy, self.fluid, -1)
        out = out - (flux[..., 1:] - flux[..., :-1]) / self.dx
        return torch.where(self.fluid, out, 0.0)

    def outflow(self):
        x, y = self.ux / self.dx, self.uy / self.dx
        return (x[..., 1:, :].clamp(min=0) - x[..., :-1, :].clamp(max=0)
                + y[..., 1:].clamp(min=0) - y[..., :-1].clamp(max=0))

    def _limited(self, c, u, fluid, axis):
        """The van Leer correction per face: only where the upwind, downwind
        and second-upwind sites are fluid sites of the grid."""
        n = c.shape[axis]

        def site(a, offset):  # the site `offset` places above each face's lower site
            pad = (3, 3) if axis == -1 else (0, 0, 3, 3)
            return torch.nn.functional.pad(a, pad).narrow(axis, 2 + offset, n + 1)

        ok = fluid.to(c.dtype)
        up_ok, dn_ok = site(ok, 0) > 0, site(ok, 1) > 0
        far_lo, far_hi = site(ok, -1) > 0, site(ok, 2) > 0
        a, b, cl, ch = site(c, 0), site(c, 1), site(c, -1), site(c, 2)

        def increment(up, down, far):
            behind, ahead = up - far, down - up
            prod = behind * ahead
            safe = torch.where(prod > 0, behind + ahead, 1.0)
            return torch.where(prod > 0, prod / safe, 0.0)

        both = up_ok & dn_ok
        plus = torch.where(both & far_lo, increment(a, b, cl), 0.0)
        minus = torch.where(both & far_hi, increment(b, a, ch), 0.0)
        return torch.where(u >= 0, u * plus, u * minus)


def _exact_transport(case, w, levels, steps, dt, ledger):
    S = levels.shape[0]
    _, xf, yf = _exact_flow(w)
    site = _Site(_t(w.obstacles, torch.bool), xf, yf, float(w.dx), case["scheme"] == "van_leer")
    diffusion = _t(DIFFUSION[:S])[:, None, None]
    low, high = torch.ones_like(diffusion), torch.zeros_like(diffusion)
    phi, fluid = _t(w.phi), site.fluid
    c = _t(levels)
    rows = []
    for _ in range(steps):
        if case.get("integration") == "crank_nicolson":
            loss = VMAX * phi / (HALF + c)

            def rate(v, loss=loss):
                return site.rate(v, diffusion, low, high) - torch.where(fluid, loss * v, 0.0)

            rhs = c + 0.5 * dt * rate(c)
            diagonal = 1.0 + 0.5 * dt * (4.0 * diffusion / float(w.dx) ** 2 + loss
                                         + site.outflow())
            first = None
            for _ in range(400):
                off = torch.where(fluid, rhs - c + 0.5 * dt * rate(c), 0.0)
                size = float(off.square().sum())
                first = size if first is None else first
                if size <= 1e-26 * first or size == 0.0:
                    break
                c = c + off / diagonal
            continue
        before = torch.where(fluid, c, 0.0)
        taken = torch.where(fluid, VMAX * phi / (HALF + c) * c, 0.0)
        moved = site.rate(c, diffusion, low, high)
        c = c + dt * (moved - taken)
        if ledger:
            volume = float(w.dx) * float(w.dy) * float(w.dz)
            after = torch.where(fluid, c, 0.0)
            rows.append(volume * torch.stack(
                [before.sum((1, 2)), after.sum((1, 2)), dt * moved.sum((1, 2)),
                 dt * taken.sum((1, 2))], 1))
    return c, torch.stack(rows) if rows else None


def _exact_coupled(case, w, seed, dt, steps):
    cells, previous = workloads.colony(w, case["cells"], seed=seed)
    _, xf, yf = _exact_flow(w)
    site = _Site(_t(w.obstacles, torch.bool), xf, yf, float(w.dx))
    diffusion = _t(DIFFUSION)[:, None, None]
    low = _t([1.0, 1.0, 1.0])[:, None, None]
    c = _t(_levels(w, 3, seed, np.float32))
    x, y = _t(cells["position_x"]) / w.dx, _t(cells["position_y"]) / w.dy
    ix, iy = x.floor().long().clamp(max=w.nx - 2), y.floor().long().clamp(max=w.ny - 2)
    fx, fy = x - ix, y - iy
    corners = [((ix + a) * w.ny + iy + b, (fx if a else 1 - fx) * (fy if b else 1 - fy))
               for a in (0, 1) for b in (0, 1)]
    length, radius = _t(cells["lengths"]), _t(cells["radii"])
    growth = _t(cells["growth_rates"])
    volume = math.pi * radius**2 * (length + 2.0 * radius)
    dilution = (_t(previous) + 2 * radius) / (length + 2 * radius)
    species = torch.ones(case["cells"], 2, dtype=torch.float64, device=_device())
    voxel = float(w.dx) * float(w.dy) * float(w.dz)
    for step in range(steps):
        flat = c.reshape(3, -1)
        seen = sum(flat[:, i] * k for i, k in corners)
        if step == 0:
            species = species * dilution[:, None]
        uptake = seen[0] / (seen[0] + 0.1) * volume
        luxi, gfp = species[:, 0], species[:, 1]
        out = torch.stack([-uptake, 0.05 * luxi * volume, 0.1 * uptake]) / voxel
        hill = seen[1] / (seen[1] + 0.5)
        species = species + dt * torch.stack(
            [2.0 * hill + 0.1 - 0.2 * luxi, growth * luxi - 0.2 * gfp], 1)
        source = torch.zeros_like(flat)
        for i, k in corners:
            source.index_add_(1, i, out * k)
        c = c + dt * (site.rate(c, diffusion, low, torch.zeros_like(low)) + source.reshape(c.shape))
    return c, species


def _exact_sweep(case, seed, dt):
    instances = _instances(case, seed)
    results = [None] * len(instances)
    masses = torch.zeros(case["steps"], len(instances), 3, dtype=torch.float64)
    for size in sorted({(i.nx, i.ny) for i in instances}):
        members = [k for k, i in enumerate(instances) if (i.nx, i.ny) == size]
        group = [instances[k] for k in members]

        def each(name):
            return _t([getattr(i, name) for i in group])

        solid = _t(np.stack([i.obstacles for i in group]).reshape(-1, *size), torch.bool)
        mobility = _t(np.stack([i.mobility for i in group]).reshape(-1, *size))
        phi = _t(np.stack([i.phi for i in group]).reshape(-1, *size))
        dx, dz = float(group[0].dx), float(group[0].dz)
        system = _Pressure(torch.where(solid, 0.0, dz * mobility), dx)
        inlet = each("inlet_pressure").float().double()
        p = system.solve(inlet)
        xf, yf = system.faces(p, solid, dz, inlet)
        site = _Site(solid, xf, yf, dx)
        diffusion = each("diffusion").float().double()[:, None, None]
        low, high = each("reservoir")[:, None, None], torch.zeros_like(diffusion)
        c = torch.zeros_like(p)
        for step in range(case["steps"]):
            taken = torch.where(site.fluid, VMAX * phi / (HALF + c) * c, 0.0)
            new = c + dt * (site.rate(c, diffusion, low, high) - taken)
            row = torch.stack([c.sum((1, 2)), new.sum((1, 2)), dt * taken.sum((1, 2))], 1)
            masses[step, members] = (row * dx * dx * dz).cpu()
            c = new
        for j, k in enumerate(members):
            results[k] = dict(x_faces=xf[j], y_faces=yf[j], levels=c[j])
    out = {name: torch.cat([r[name].reshape(-1) for r in results]).cpu().numpy()
           for name in results[0]}
    out["masses"] = masses.numpy()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "resolved":
        return None  # a saddle-point system without a quick dense solution
    if kind == "sweep":
        state = prepare(case, seed)
        state["hip"].close()
        return _exact_sweep(case, seed, float(np.float32(state["dt"])))
    w = _geometry(case, seed)

    def flat(a):
        return a.reshape(-1).cpu().numpy()

    if kind in ("call", "solve"):
        _, x, y = _exact_flow(w)
        return dict(x_faces=flat(x), y_faces=flat(y), z_faces=np.zeros(2 * w.nx * w.ny))
    state = prepare(case, seed)
    state["hip"].close()
    dt = float(np.float32(state["dt"]))
    if kind == "coupled":
        levels, species = _exact_coupled(case, w, seed, dt, case["steps"])
        return dict(levels=flat(levels), species=flat(species))
    dtype = np.float64 if case.get("precision") == 64 else np.float32
    ledger = kind == "transport" and state["ledger"]
    levels, rows = _exact_transport(case, w, _levels(w, case["signals"], seed, dtype),
                                    case.get("steps", 1), dt, ledger)
    out = dict(levels=flat(levels))
    if ledger:
        out["ledger"] = rows.cpu().numpy()
    return out
