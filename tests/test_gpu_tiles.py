"""The object tile kernels and the probe sums at the edges of their splits, against the FP64
oracle in complex128: an object of more tiles than the split takes and of fewer, batches of more
and fewer views than it needs there, one where the gathers are split and the overlaps are not, tiles
with more views than one round stages (256), one mode and an odd number, and chunk counts of the
probe sums on both sides of their own split. 1e-9 is the complex128 bound of the other parity tests:
the splits only regroup sums of at most 300 terms (300·2^-53 = 3e-14)."""

import math

import numpy as np
import pytest

from conftest import max_rel
from test_gpu_lsqml import run_oracle
from test_gpu_rpie import gpu, oracle, rel_l2
from ptyrs_amd import sim

pytestmark = pytest.mark.gpu

# frame side, modes, frames, object (rows, columns): 10 tiles of 300 views each; 20 tiles; 1000
# tiles, whose gathers split from 20 views on and overlaps from 77; more tiles than are split, the
# last column and row of them ragged.
CASES = [(16, 1, 300, (40, 40)), (16, 3, 20, (40, 72)), (32, 3, 24, (500, 500)),
         (32, 3, 12, (1042, 500))]
TILES = [math.ceil(c[3][0] / 4) * math.ceil(c[3][1] / 64) for c in CASES]
assert TILES == [10, 20, 1000, 2088]


def scan(case):
    n, modes, frames, side = case
    pixel = sim.pixel_size(n)
    rng = np.random.default_rng(11)
    y, x = rng.uniform(-1, 1, (2, frames))
    y, x = (v - v.mean() for v in (y, x))  # the scan is centred on its mean
    y, x = (v / np.abs(v).max() * ((s - n) / 2 - 4) * pixel for v, s in zip((y, x), side))
    obj = sim.random_object(*side, 3)
    probe = sim.hermite_gauss_probe(n, powers=[0.8, 0.2, 0.05][:modes])
    cy, cx = sim.corners(y, x, pixel, side, n)
    intensity = sim.intensities(obj, probe, cy, cx, sim.quad_phase(n))
    s = 2e5 / intensity.sum(axis=(1, 2)).mean()
    start = np.exp(1j * rng.uniform(-1.0, 1.0, obj.shape))
    return dict(counts=rng.poisson(intensity * s).astype(np.float32), y=y, x=x, obj=start,
                probe=probe * math.sqrt(s) * 0.9)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("name,kw", [("rpie", dict(batch_size=300)), ("rpie", dict(batch_size=7)),
                                     ("rpie", dict(batch_size=3)),
                                     ("ap", dict(probe_inertia=0.001)),
                                     ("ml", dict(update_probe=True))])
def test_tiles(case, name, kw):
    d = scan(case)
    g, o = gpu(d, "c128"), oracle(d)
    getattr(g, name)(2, calc_llk=1, **kw)
    getattr(o, name)(2, calc_llk=1, **kw)
    assert max_rel(g.history["poisson"], [r[2].poisson for r in o.history]) < 1e-8
    assert rel_l2(g.object, o.obj) < 1e-8
    assert rel_l2(g.probe, o.probe) < 1e-8


@pytest.mark.parametrize("case", CASES)
def test_tiles_lsqml(case):
    d = scan(case)
    g, o = gpu(d, "c128"), oracle(d)
    batch = case[2]
    obj, probe, llks, _ = run_oracle(o, 2, batch, "poisson", 5)
    g.lsqml(2, 1, batch, "poisson", 5)
    assert max_rel(g.history["poisson"], llks) < 1e-8
    assert rel_l2(g.object - d["obj"], obj - d["obj"]) < 1e-8
    assert rel_l2(g.probe - d["probe"], probe - d["probe"]) < 1e-8
