"""The object-plane line transforms at sides whose plans differ: powers of two alone, a radix 3,
odd radices on both sides of the matrix products' 16-row tiles (5, 7, 11, 31, 37), two odd radices
in one plan, a repeated one, a prime side, different plans on the two axes. The sampled model
intensities and one rPIE epoch (windows, their adjoint, the overlaps) against the FP64 oracle.
complex64: a line's transform is within 3e-7 of its norm at these radices, the intensities take
four of them."""

import numpy as np
import pytest

from test_gpu_rpie import gpu, oracle, rel_l2, small_scan

pytestmark = pytest.mark.gpu

SIDES = [(64, 64), (48, 50), (49, 56), (55, 66), (62, 74), (75, 70), (61, 63)]


@pytest.mark.parametrize("dtype,tol", [("c128", 1e-11), ("c64", 1e-5)])
@pytest.mark.parametrize("side", SIDES)
def test_sampled_windows_at_every_plan(side, dtype, tol):
    d = small_scan(n=32, nprobe=2, npos=9, masked=False)
    d["y"], d["x"] = d["y"] * 0.4, d["x"] * 0.4  # the frames stay inside every side
    rng = np.random.default_rng(2)
    d["obj"] = np.exp(1j * rng.uniform(-1.0, 1.0, (1, *side)))
    d0 = rng.uniform(-0.45, 0.45, (9, 2))
    g, o = gpu(d, dtype), oracle(d)
    for e in (g, o):
        e.set_sampling("full_object")
    o.set_position(d0, refine=False)
    g.set_features(position=d0, hold=("position",))
    start = d["obj"]
    kw = dict(batch_size=4, calc_llk=1, seed=5)
    g.rpie(1, **kw)
    o.rpie(1, **kw)
    assert rel_l2(g.object - start, o.obj - start) < 10 * tol
    assert abs(g.history["poisson"][0] / o.history[0][2].poisson - 1) < tol
