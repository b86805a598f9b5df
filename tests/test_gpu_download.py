"""The state comes back exactly as it was set, at array sizes around the download's pieces: below
its ring, a piece short of and past its first thread, a ragged last piece, several pieces per
worker; the ring is made by the larger arrays and used by the smaller ones after them."""

import numpy as np
import pytest

import ptyrs_amd as pa
from ptyrs_amd import sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["c64", "c128"])
@pytest.mark.parametrize("sides", [[(70, 90), (723, 725), (300, 501)], [(1024, 512), (1025, 1023)],
                                   [(1500, 1503), (363, 362)]])
def test_state_round_trip(dtype, sides):
    rng = np.random.default_rng(4)
    n = 64
    for ny, nx in sides:
        obj = rng.normal(size=(1, ny, nx)) + 1j * rng.normal(size=(1, ny, nx))
        probe = rng.normal(size=(2, n, n)) + 1j * rng.normal(size=(2, n, n))
        scan = pa.Scan(np.ones((1, n, n), np.float32), [0.0], [0.0], sim.WAVELENGTH, sim.DISTANCE,
                       sim.DETECTOR_PIXEL)
        g = pa.GpuPtycho(scan, obj, probe, dtype=dtype)
        for a in (obj, 2 * obj):
            g.set_object(a)
            want = a.astype(np.complex64) if dtype == "c64" else a
            np.testing.assert_array_equal(g.object, want[0] if g.object.ndim == 2 else want)
        want = probe.astype(np.complex64) if dtype == "c64" else probe
        np.testing.assert_array_equal(g.probe, want)
