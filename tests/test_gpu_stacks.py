"""AP, ML and DM with a short last stack that alone would be cut into more chunks than a full
stack (128 frames, or a stack size of its own): every frame's probe partial is in the update.
Against the FP64 oracle, with the bounds of the other parity tests; five frames of 176 left out
move the probe by percents."""

import pytest

from conftest import max_rel
from test_gpu_rpie import gpu, oracle, rel_l2, small_scan

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-9, "c64": 1e-4}


@pytest.mark.parametrize("dtype,n,nprobe,npos,stack", [
    ("c64", 128, 2, 176, None), ("c64", 128, 1, 208, None), ("c64", 64, 4, 198, None),
    ("c128", 64, 2, 198, None), ("c64", 128, 2, 104, 64)])
@pytest.mark.parametrize("name", ["ap", "ml"])
def test_short_last_stack(name, dtype, n, nprobe, npos, stack):
    d = small_scan(n=n, nprobe=nprobe, npos=npos)
    g, o = gpu(d, dtype, **(dict(stack_size=stack) if stack else {})), oracle(d)
    kw = dict(probe_inertia=0.001) if name == "ap" else dict(update_probe=True)
    check(g, o, dtype, name, kw)


def test_short_last_stack_dm():
    d = small_scan(n=64, nprobe=5, npos=218)
    check(gpu(d, "c64"), oracle(d), "c64", "dm", {})


def check(g, o, dtype, name, kw):
    getattr(g, name)(2, calc_llk=1, **kw)
    getattr(o, name)(2, calc_llk=1, **kw)
    tol = TOL[dtype]
    assert max_rel(g.history["poisson"], [r[2].poisson for r in o.history]) < tol
    assert rel_l2(g.object, o.obj) < tol * (10 if dtype == "c128" else 30)
    assert rel_l2(g.probe, o.probe) < tol * (10 if dtype == "c128" else 30)
