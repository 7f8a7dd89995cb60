"""Device memory of the adaptive octree's working sets: no more than sorting them takes."""
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds
from mlodsurfaces_amd import hiprt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [7, 8, 9])
def test_bytes_a_leaf(depth):
    w = ds.make_workload("torus1m")
    t = A.APSSOctree().build(ds.pn_normalize(w["points"])[::4], w["normals"][::4])
    ap = A.Fastapss(t, A.Kernel(**w["kernel"]))
    ap.setScalingProtectionSphere(w["cutoff"])
    ap.set_precision("fp32c")
    A.OctreeGenerator(ap, ap._kernel).generate(depth)  # the runtime's own, and the tree's query buffers
    A.trim_memory()
    free0, _ = hiprt.mem_info()
    g = A.OctreeGenerator(ap, ap._kernel)
    leaves = len(g.generate(depth))
    A.trim_memory()
    held = free0 - hiprt.mem_info()[0]
    # 900 bytes a leaf with every set sorted; what is left over at small sizes is the least size of the vectors
    assert held <= 900 * leaves + (24 << 20)
    g.close()
