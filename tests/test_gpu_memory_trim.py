"""The library's kept device memory goes back when asked for, and work goes on after it."""
import numpy as np
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds
from mlodsurfaces_amd import hiprt

pytestmark = pytest.mark.gpu


def _project(p, n, q):
    t = A.APSSOctree().build(p, n)
    ap = A.Fastapss(t, A.Kernel(type=2, sigmas=[0.05, 0.1]))
    ap.set_precision("fp32c")
    out = ap.project_points(q, 2)
    held = t.info()["device_bytes"]
    t.free()
    return out, held


def test_trim_gives_the_memory_back():
    p, n = ds.sphere(1_500_000, seed=5)
    q = p[:1000]
    _project(p, n, q)  # the runtime's own: code, staging of copies of this size
    A.trim_memory()
    free0, total = hiprt.mem_info()
    ref, held = _project(p, n, q)
    kept = free0 - hiprt.mem_info()[0]
    assert kept > held // 2 > 32 << 20  # (held fits the bound)
    A.trim_memory()
    assert abs(free0 - hiprt.mem_info()[0]) <= 4 << 20
    got, _ = _project(p, n, q)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
    A.trim_memory()


def test_device_bytes_are_whole_blocks():
    """Every block of a tree is a multiple of its size class's step, an eighth of the power of two below it."""
    for m in (10, 1000, 100_000):
        p, n = ds.sphere(m, seed=6)
        t = A.APSSOctree().build(p, n)
        i = t.info()
        asked = i["n_nodes"] * (16 + 16 + 64 + 64 + 64 + 8 + 24 + 8) + m * (16 + 16 + 4 + 4)
        assert asked <= i["device_bytes"] <= max(1.125 * asked + 4096 * 12, asked)
        assert i["device_bytes"] % 256 == 0
        t.free()
