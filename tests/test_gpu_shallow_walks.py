"""Trees of one leaf and of one level, where leaves of several points are all there is: the lane, grouped and wave walks
against one another, and against the oracle (REF_CPU keeps one point of a leaf: no sphere there, and the walks alone
are compared)."""
import numpy as np
import pytest

from gpu_util import gpu_project, gpu_tree
from mlodsurfaces_amd import datasets as ds

pytestmark = pytest.mark.gpu

K = dict(type=2, sigmas=[0.1, 0.2, 0.4])


@pytest.mark.parametrize("max_depth,leaf,min_depth", [(1, 1, 0), (1, 1, 1), (2, 1, 1), (12, 3000, 0), (12, 3000, 2), (12, 500, 0)])
@pytest.mark.parametrize("semantics", ["ref_gpu", "ref_cpu"])
@pytest.mark.parametrize("precision", ["fp32", "fp32c", "fp64"])
def test_walks_agree(oracle_built, max_depth, leaf, min_depth, semantics, precision):
    p, n = ds.torus(2000, seed=121)
    t = gpu_tree(p, n, maxDepth=max_depth, maxNumberOfPointsPerLeaf=leaf)
    q = ds.jitter_queries(p[:300], 0.05, seed=122)
    kw = dict(cutoff=2.0, min_depth=min_depth, semantics=semantics, precision=precision)
    a = gpu_project(t, q, K, **kw)[:2]
    b = gpu_project(t, np.tile(q, (200, 1)), K, **kw)[:2]
    w = gpu_project(t, q, K, traversal="wave", **kw)[:2]
    for x, y, z in zip(a, b, w):
        assert np.array_equal(x.view(np.int32), y[:300].view(np.int32))
        if precision == "fp64":
            assert np.array_equal(x, z)
    if semantics == "ref_gpu" and precision != "fp32":
        o = oracle_built.OracleTree(p, n, max_depth=max_depth, max_pts_per_leaf=leaf)
        op, on = o.project(q, oracle_built.make_kernel(**K),
                           oracle_built.make_params(cutoff=2.0, min_depth=min_depth, semantics=semantics), precision=1)
        assert np.abs(a[0] - op).max() <= 1e-6 * 2 * ds.bbox_radius(p) and np.abs(a[1] - on).max() <= 1e-5

