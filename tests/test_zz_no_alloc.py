"""The allocation-free transport step (msim_hip_advance_signal_grid_static)
against msim_hip_advance_signal_grid, through the C ABI.

The static entry point stages everything in one file-scope device array and
allocates nothing; its results must equal the allocating entry point's bit for
bit (FP32 levels), on two calls in a row whose second grid is smaller, so the
second call runs over what the first left in the array.
"""
from __future__ import annotations

import numpy as np
import pytest

import microsimulator_amd as msa
from tests.helpers import FIXED, NO_FLUX, PERIODIC, random_transport_case

pytestmark = pytest.mark.gpu

KINDS = (FIXED, FIXED, PERIODIC, PERIODIC, NO_FLUX, NO_FLUX)


def _spec(nx, ny, S, seed, scheme, reaction):
    c = random_transport_case(nx, ny, S, KINDS, seed)
    grid = msa.Grid(nx, ny, 1, 1.0, 1.0, 1.0, c["solid"], KINDS)
    kw = {}
    if reaction == "affine":
        kw = dict(loss_rates=c["loss"], source_rates=c["source"])
    elif reaction == "monod":
        kw = dict(phi=c["phi"], monod_vmax=np.full(S, 0.3, np.float32),
                  monod_k=np.full(S, 0.5, np.float32))
    spec = msa.SignalGridSpec(grid, c["diffusion"], c["bv"],
                              msa.VelocityField(c["xf"], c["yf"], c["zf"]),
                              advection_scheme=scheme, **kw)
    return spec, c["levels"].astype(np.float32)


@pytest.mark.parametrize("scheme,reaction", [(msa.UPWIND, "monod"), (msa.VAN_LEER, "affine"),
                                             (msa.UPWIND, None)])
def test_static_step_equals_the_allocating_step(hip, scheme, reaction):
    # Two calls in a row: the second grid is smaller and has fewer signals.
    for nx, ny, S, seed in ((300, 260, 3, 11), (70, 45, 2, 12)):
        spec, levels = _spec(nx, ny, S, seed, scheme, reaction)
        print(f"static step: {nx}x{ny}, {S} signals, scheme {scheme}, {reaction}", flush=True)
        dt = 0.02
        ref, ref_rep = hip.advance_signal_grid(spec, levels, dt)
        got, rep = hip.advance_signal_grid_static(spec, levels, dt)
        assert np.array_equal(got, ref)
        assert rep == ref_rep
        # A second step from the result, as a caller's loop takes it.
        ref2, _ = hip.advance_signal_grid(spec, ref, dt)
        got2, _ = hip.advance_signal_grid_static(spec, got, dt)
        assert np.array_equal(got2, ref2)


def test_static_step_refuses_what_the_allocating_step_refuses(hip):
    spec, levels = _spec(64, 48, 2, 21, msa.UPWIND, "affine")
    # The explicit bound, with the reference's message.
    with pytest.raises(msa.InvalidArgument, match="explicit stability bound"):
        hip.advance_signal_grid_static(spec, levels, 50.0)
    with pytest.raises(msa.InvalidArgument, match="explicit stability bound"):
        hip.advance_signal_grid(spec, levels, 50.0)
    # A negative level.
    bad = levels.copy()
    bad[np.argmax(bad)] = -1.0
    with pytest.raises(msa.InvalidArgument, match="finite and non-negative"):
        hip.advance_signal_grid_static(spec, bad, 0.02)
    # After refusals the next call still equals the allocating step.
    ref, _ = hip.advance_signal_grid(spec, levels, 0.02)
    got, _ = hip.advance_signal_grid_static(spec, levels, 0.02)
    assert np.array_equal(got, ref)


def test_static_step_limits(hip):
    lib = msa.library()
    limit = int(lib.msim_hip_static_scratch_bytes())
    assert limit == 64 << 20
    # A grid whose two level buffers alone exceed the scratch is refused
    # before any device work.
    nx, ny, S = 2048, 2048, 3
    grid = msa.Grid(nx, ny, 1, 1.0, 1.0, 1.0, None, KINDS)
    spec = msa.SignalGridSpec(grid, np.full(S, 0.1, np.float32))
    with pytest.raises(msa.InvalidArgument, match="bytes of device scratch"):
        hip.advance_signal_grid_static(spec, np.zeros(S * nx * ny, np.float32), 0.1)
    # Implicit steps and reservoir patches are the allocating entry point's.
    small, levels = _spec(32, 24, 1, 5, msa.UPWIND, None)
    small.integration = msa.CRANK_NICOLSON
    with pytest.raises(msa.Unsupported):
        hip.advance_signal_grid_static(small, levels, 0.1)


def _scratch(nx, ny, S, scheme):
    """Bytes a field-less step over nx x ny sites takes of the scratch array:
    strips of at most 254 columns (252 under van Leer) by 16 x-rows (or fewer,
    down to 4, for 2048 blocks), 49 doubles a block, and the staged mask and
    levels."""
    halo = 4 if scheme == msa.VAN_LEER else 2
    strips = min((-(-ny // (t - halo)) * t, -(-ny // (t - halo))) for t in (256, 128, 64))[1]
    rows = 16
    while rows > 4 and strips * -(-nx // rows) < 2048:
        rows //= 2
    blocks = max(strips * -(-nx // rows), 24)
    survey = min(-(-nx * ny // 256), 2048)
    regions = [176, 12, 64, 8 * max(49 * blocks, 9 * survey), nx * ny, 4 * S * nx * ny,
               4 * S * nx * ny]
    return sum(-(-r // 256) * 256 for r in regions)


@pytest.mark.parametrize("nx,scheme", [(1, msa.UPWIND), (3, msa.VAN_LEER), (4, msa.UPWIND),
                                       (5, msa.VAN_LEER), (40, msa.UPWIND)])
def test_static_step_takes_what_the_scratch_array_holds(hip, nx, scheme):
    """The widest grid that fits is taken, one column more refused, also where a
    grid has more walks than the blocks the array has partials for."""
    limit = hip.lib.msim_hip_static_scratch_bytes()
    lo, hi = 1, limit // nx
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if _scratch(nx, mid, 1, scheme) <= limit else (lo, mid)

    def step(ny, entry):
        levels = np.random.default_rng(ny).random(nx * ny).astype(np.float32)
        spec = msa.SignalGridSpec(msa.Grid(nx, ny, 1, 1.0, 1.0, 1.0, None, KINDS),
                                  np.ones(1, np.float32), np.zeros(6, np.float32),
                                  advection_scheme=scheme)
        return entry(spec, levels, 0.1)[0]

    assert np.array_equal(step(lo, hip.advance_signal_grid_static),
                          step(lo, hip.advance_signal_grid))
    with pytest.raises(msa.InvalidArgument, match="bytes of device scratch"):
        step(lo + 1, hip.advance_signal_grid_static)
