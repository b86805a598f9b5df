"""The state comes back exactly as it was set, at array sizes around the download's pieces: below
its ring, a piece short of and past its first helper, a ragged last piece, several pieces per
thread. Each state is read several times; the ring is made by an object of at least 4 MB, and the
probe of four modes of 256² (2 MB in complex64, 4 in complex128) goes through it after that."""

import numpy as np
import pytest

import ptyrs_amd as pa
from ptyrs_amd import sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["c64", "c128"])
@pytest.mark.parametrize("side", [(270, 290), (723, 725), (300, 501), (1024, 512), (1025, 1023),
                                  (1500, 1503), (363, 362)])
def test_state_round_trip(dtype, side):
    rng = np.random.default_rng(4)
    n = 256
    obj = rng.normal(size=(1, *side)) + 1j * rng.normal(size=(1, *side))
    probe = rng.normal(size=(4, n, n)) + 1j * rng.normal(size=(4, n, n))
    scan = pa.Scan(np.ones((1, n, n), np.float32), [0.0], [0.0], sim.WAVELENGTH, sim.DISTANCE,
                   sim.DETECTOR_PIXEL)
    g = pa.GpuPtycho(scan, obj, probe, dtype=dtype)
    single = (lambda a: a.astype(np.complex64)) if dtype == "c64" else (lambda a: a)
    for k in range(1, 5):
        g.set_object(k * obj)
        want = single(k * obj)
        np.testing.assert_array_equal(g.object, want[0] if g.object.ndim == 2 else want)
        np.testing.assert_array_equal(g.probe, single(probe))
