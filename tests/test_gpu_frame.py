"""rPIE where a frame runs in one workgroup (complex64, sides 32 to 64, one mode) and beside it (more
modes), with both arrays updated and with either held, masked pixels, one frame a
batch and batches that do not divide the scan, against the FP64 oracle. The bounds are those of
the other complex64 runs of rPIE: the operations and their order per pixel are the stack's. One
frame a batch runs at 64: at 32 with one mode it amplifies a rounding 4e4-fold in two epochs
(complex128 1e-16 to 5e-12, the stack's complex64 6e-8 to 8e-4), which no bound here can hold."""

import numpy as np
import pytest
import torch

from ptyrs_amd import sim
from test_gpu_rpie import TOL, gpu, oracle, rel_l2, small_scan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(), dict(probe_step=None), dict(obj_step=None)])
@pytest.mark.parametrize("n,nprobe,batch", [(64, 1, 1), (64, 1, 30), (64, 1, 7), (32, 1, 7),
                                            (48, 1, 13), (32, 4, 7), (48, 2, 7), (64, 3, 7)])
def test_rpie_frames(n, nprobe, batch, kw):
    d = small_scan(n=n, nprobe=nprobe, npos=30)
    g, o = gpu(d, "c64"), oracle(d)
    p = dict(batch_size=batch, calc_llk=1, seed=5, **kw)
    g.rpie(2, **p)
    o.rpie(2, **p)
    assert rel_l2(g.object, o.obj) < TOL["c64"] * 10
    assert rel_l2(g.probe, o.probe) < TOL["c64"] * 10
    want = [r[2].poisson for r in o.history]
    assert all(abs(a / b - 1) < TOL["c64"] for a, b in zip(g.history["poisson"], want))


def test_large_batch_holds_no_second_stack():
    """A batch past the frames' own probe directions (4096) holds the stack's exit waves and, beside
    them, less than half as much again."""
    n, frames = 64, 12000
    rng = np.random.default_rng(8)
    y, x = rng.uniform(-20, 20, (2, frames)) * sim.pixel_size(n)
    obj = np.exp(1j * rng.uniform(-1.0, 1.0, (1, 128, 128)))
    probe = sim.hermite_gauss_probe(n, powers=[1.0]) * 100
    g = gpu(dict(counts=np.ones((frames, n, n), np.float32), y=y, x=x, obj=obj, probe=probe), "c64")
    free = torch.cuda.mem_get_info()[0]
    g.rpie(1, batch_size=frames)
    assert free - torch.cuda.mem_get_info()[0] < 1.5 * frames * n * n * 8
    assert np.isfinite(g.object).all()
