"""The explicit transport step at the edges of its strips (62 columns per wave,
60 under van Leer) and walks (1, 2, 4, 8 or 12 x-rows), FP32 bit for bit with the
oracle, which is bit-exact with the reference, and FP64 to 1e-13 relative."""
import numpy as np
import pytest

import microsimulator_amd as msa
from oracle import VAN_LEER
from oracle import Grid as OGrid
from tests.helpers import FIXED, NO_FLUX, PERIODIC, random_transport_case
from tests.test_gpu_implicit import oracle_kw, same_report, spec_of

pytestmark = pytest.mark.gpu

KINDS = [(FIXED, FIXED, NO_FLUX, FIXED, NO_FLUX, NO_FLUX),
         (PERIODIC, PERIODIC, PERIODIC, PERIODIC, NO_FLUX, NO_FLUX),
         (NO_FLUX, FIXED, FIXED, NO_FLUX, NO_FLUX, NO_FLUX)]


@pytest.mark.parametrize("kinds", KINDS)
@pytest.mark.parametrize("limited", [False, True])
@pytest.mark.parametrize("shape,S", [
    ((4, 59), 1), ((5, 60), 3), ((3, 61), 1), ((13, 62), 2), ((11, 63), 3), ((12, 64), 8),
    ((25, 119), 1), ((7, 121), 2), ((6, 124), 5), ((9, 125), 1), ((2, 2), 1), ((1, 63), 1),
    ((1500, 61), 1), ((2300, 187), 1), ((3101, 61), 1), ((3071, 63), 2), ((8195, 63), 1),
    ((16399, 64), 1),
])
def test_step_at_strip_edges(hip, oracle, shape, S, limited, kinds):
    nx, ny = shape
    d = random_transport_case(nx, ny, S, kinds, seed=7 * nx + ny)
    og = OGrid(nx, ny, 1, 1.0, 0.5, 1.0, d["solid"], kinds)
    kw = dict(diffusion=d["diffusion"], boundary_values=d["bv"],
              faces=np.concatenate([d["xf"], d["yf"], d["zf"]]))
    spec = msa.SignalGridSpec(msa.Grid(nx, ny, 1, 1.0, 0.5, 1.0, d["solid"], kinds),
                              d["diffusion"], d["bv"],
                              msa.VelocityField(d["xf"], d["yf"], d["zf"]))
    if S != 3:  # with Monod uptake
        spec.phi, spec.monod_vmax, spec.monod_k = d["phi"], [0.7] * S, [0.2] * S
        kw.update(phi=d["phi"], vmax=[0.7] * S, monod_k=[0.2] * S)
    if limited:
        spec.advection_scheme, kw["scheme"] = msa.VAN_LEER, VAN_LEER
    lv32 = d["levels"].astype(np.float32)
    hip.adr_upload(spec, lv32, precision=32)
    hip.adr_run(0.02, 4, ledger=False)
    ref = oracle.adr_step_f32(og, lv32, 0.02, steps=4, **kw)
    assert np.array_equal(hip.adr_download(), ref)
    if S <= 3:
        one, _ = hip.advance_signal_grid_static(spec, lv32, 0.02)
        assert np.array_equal(one, oracle.adr_step_f32(og, lv32, 0.02, **kw))
    hip.adr_upload(spec, d["levels"], precision=64)
    ledger = hip.adr_run(0.02, 4)
    ref64, ref_ledger = oracle.adr_step_f64(og, d["levels"], 0.02, steps=4, **kw)
    assert np.abs(hip.adr_download() - ref64).max() <= 1e-13 * np.abs(ref64).max()
    # Supply and uptake in proportion to the mass they are added to (1e-12 of
    # it, 1e-13 per step's own rounding times its sums).
    scale = np.abs(ref_ledger[:, :, 1:2])
    assert (np.abs(ledger - ref_ledger) <= 1e-12 * scale + 1e-300).all()


def test_settle_of_a_marked_step(hip, oracle):
    """A front carried into empty fluid by van Leer leaves levels below zero by
    rounding on some steps and none on others: the settle that only runs over
    the levels of a marked step gives the oracle's levels after every step."""
    nx, ny = 90, 130
    rng = np.random.default_rng(3)
    xf = np.full((nx + 1, ny), 0.73, np.float32)
    grid = msa.Grid(nx, ny, 1, 1.0, 1.0, 1.0, None,
                    (FIXED, FIXED, NO_FLUX, NO_FLUX, NO_FLUX, NO_FLUX))
    zero_y, zero_z = np.zeros(nx * (ny + 1), np.float32), np.zeros(2 * nx * ny, np.float32)
    levels = np.zeros((nx, ny), np.float32)
    levels[10:30] = rng.random((20, ny)).astype(np.float32)
    spec = msa.SignalGridSpec(grid, np.zeros(1, np.float32), np.zeros(6, np.float32),
                              msa.VelocityField(xf.reshape(-1), zero_y, zero_z),
                              advection_scheme=msa.VAN_LEER)
    og = OGrid(nx, ny, 1, 1.0, 1.0, 1.0, None, grid.boundary)
    ref = levels.reshape(-1)
    hip.adr_upload(spec, ref, precision=32)
    for _ in range(40):
        hip.adr_run(0.6, 1, ledger=False)
        ref = oracle.adr_step_f32(og, ref, 0.6, diffusion=[0.0], scheme=VAN_LEER,
                                  boundary_values=np.zeros(6, np.float32),
                                  faces=np.concatenate([xf.reshape(-1), zero_y, zero_z]))
        assert np.array_equal(hip.adr_download(), ref)
    assert ref.min() >= 0.0


@pytest.mark.parametrize("limited", [False, True])
@pytest.mark.parametrize("shape,kinds", [((13, 62), KINDS[0]), ((5, 61), KINDS[1]),
                                         ((30, 125), KINDS[2]), ((1400, 63), KINDS[0]),
                                         ((1, 130), KINDS[2]), ((3101, 61), KINDS[1]),
                                         ((3071, 63), KINDS[0]), ((2067, 121), KINDS[1]),
                                         ((8195, 63), KINDS[2]), ((16399, 64), KINDS[0])])
def test_implicit_steps_at_strip_edges(hip, oracle, shape, kinds, limited):
    """Several implicit steps on the device (the accepted iterate changes
    buffers from step to step by its parity) bit for bit with the oracle's,
    obstacle levels included; walks of 1, 2, 4 and 8 rows with ragged ends."""
    nx, ny = shape
    c = random_transport_case(nx, ny, 2, kinds, seed=3 * nx + ny)
    scheme = msa.VAN_LEER if limited else msa.UPWIND
    og = OGrid(nx, ny, 1, 1.0, 0.5, 1.0, c["solid"], kinds)
    spec = spec_of(msa.Grid(nx, ny, 1, 1.0, 0.5, 1.0, c["solid"], kinds), c, scheme,
                   msa.CRANK_NICOLSON)
    ref = c["levels"].astype(np.float32)
    hip.adr_upload(spec, ref, precision=32)
    for dt in (0.02, 0.3, 0.1, 0.01):
        hip.adr_run(dt, 1, ledger=False)
        ref, rep = oracle.adr_step_implicit(og, ref, dt,
                                            **oracle_kw(c, scheme, msa.CRANK_NICOLSON))
        assert np.array_equal(hip.adr_download(), ref)
        same_report(hip.adr_report(), rep)
