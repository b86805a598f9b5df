"""The probe's sums over slots and chunks where the pixels and modes leave 8, 2, 2 and 1 thread
groups a workgroup (smaller frames have 16), fewer slots than groups among them, against the FP64
oracle in complex128: the gradient, AP's probe, and the frames' directions moved back under position
offsets. 1e-9 is the bound of the other parity tests; the groups only regroup sums of a few terms."""

import numpy as np
import pytest

from oracle.lsqml import POISSON, cost_grads
from test_gpu_rpie import gpu, oracle, rel_l2, small_scan

pytestmark = pytest.mark.gpu

SHAPES = [(256, 1, 5), (256, 3, 9), (512, 1, 5), (512, 2, 3)]


@pytest.mark.parametrize("n,nprobe,npos", SHAPES)
def test_gradient(n, nprobe, npos):
    d = small_scan(n=n, nprobe=nprobe, npos=npos)
    g, o = gpu(d, "c128"), oracle(d)
    v, go, gp = g.grad("poisson")
    wv, wo, wp = cost_grads(o.optics, o.views_all, o.iobs, o.addr.nmode, o.obj, o.probe, POISSON)
    assert abs(v - wv) <= 1e-9 * abs(wv)
    assert rel_l2(go[0], wo) < 1e-8 and rel_l2(gp, wp) < 1e-8


@pytest.mark.parametrize("n,nprobe,npos", SHAPES)
def test_projection_probe(n, nprobe, npos):
    d = small_scan(n=n, nprobe=nprobe, npos=npos)
    g, o = gpu(d, "c128"), oracle(d)
    g.ap(2, probe_inertia=0.001)
    o.ap(2, probe_inertia=0.001)
    assert rel_l2(g.object, o.obj) < 1e-8 and rel_l2(g.probe, o.probe) < 1e-8


@pytest.mark.parametrize("n,nprobe,npos", SHAPES)
def test_moved_directions(n, nprobe, npos):
    d = small_scan(n=n, nprobe=nprobe, npos=npos)
    d0 = np.random.default_rng(31).uniform(-0.4, 0.4, (npos, 2))
    g, o = gpu(d, "c128"), oracle(d)
    o.set_position(d0, refine=True)
    g.set_features(position=d0)
    kw = dict(batch_size=npos, calc_llk=1, seed=5)
    g.rpie(2, **kw)
    o.rpie(2, **kw)
    assert rel_l2(g.object, o.obj) < 1e-8 and rel_l2(g.probe, o.probe) < 1e-8
