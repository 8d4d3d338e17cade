"""Large results through the pinned slots: every byte arrives, whatever the
size against the slot (2 MiB) and the threaded path's threshold (4 MiB), also
from several contexts at once, and again after the last context is gone."""
import threading

import numpy as np
import pytest

import microsimulator_amd as msa

pytestmark = pytest.mark.gpu

KINDS = (msa.FIXED, msa.FIXED, msa.NO_FLUX, msa.NO_FLUX, msa.NO_FLUX, msa.NO_FLUX)


def round_trip(hip, nx, ny, seed):
    levels = np.random.default_rng(seed).random(nx * ny).astype(np.float32)
    spec = msa.SignalGridSpec(msa.Grid(nx, ny, 1, 1.0, 1.0, 1.0, None, KINDS),
                              np.ones(1, np.float32))
    hip.adr_upload(spec, levels, precision=32)
    return np.array_equal(hip.adr_download(), levels)


@pytest.mark.parametrize("nx,ny", [
    (3, 5), (1023, 1024), (1024, 1024), (1025, 1024), (1, (1 << 20) + 1), (1531, 769),
    (2048, 1536), (2047, 1537), (4096, 4099),
])
def test_download_sizes(nx, ny):
    with msa.HipBackend(0) as hip:
        assert round_trip(hip, nx, ny, nx + ny)
        assert round_trip(hip, nx, ny, nx)


def test_download_from_several_contexts():
    results = []

    def work(k):
        with msa.HipBackend(0) as hip:
            results.extend(round_trip(hip, 1200 + 17 * k, 1311, 10 * k + j) for j in range(3))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 12 and all(results)
    with msa.HipBackend(0) as hip:
        assert round_trip(hip, 1500, 1400, 5)
