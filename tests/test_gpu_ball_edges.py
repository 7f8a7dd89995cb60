"""Ball APSS on the matrix cores: ranges at the edges of a 64-point load and of a 512-point subtree, query counts at
the edges of a wavefront's 16, balls that hold every point, few, or none, against the FP64 oracle."""
import numpy as np
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds
from oracle import bind

pytestmark = pytest.mark.gpu

SIG = [0.2, 0.4]


def _plugin(p, n, r, precision, **kw):
    t = A.APSSOctree().build(p, n, **kw)
    t.ballMode(True, r)
    ap = A.Fastapss(t, A.Kernel(type=2, sigmas=SIG))
    ap.set_precision(precision)
    ap.set_semantics("ref_cpu")
    return ap


@pytest.mark.parametrize("n", [20, 63, 64, 65, 511, 512, 513, 3000])
@pytest.mark.parametrize("r", [0.4, 5.0])  # some of the points; all of them
def test_range_sizes(n, r):
    p, nr = ds.sphere(n, seed=51, noise=0.02)
    q = np.concatenate([ds.jitter_queries(p[:20], 0.03, seed=52), p[:5], [[9.0, 9.0, 9.0]]]).astype(np.float32)
    o = bind.OracleTree(p, nr)
    op, on = o.project(q, bind.make_kernel(type=2, sigmas=SIG),
                       bind.make_params(cutoff=2.0, semantics="ref_cpu", mode="ball", ball_radius=r), precision=1)
    cnt = (np.linalg.norm(p[None].astype(np.float64) - q[:, None], axis=2) <= r).sum(1)
    keep = cnt >= 8  # fewer points do not determine a sphere
    assert (keep.sum() >= 3 or n < 500) and cnt[-1] == 0
    for precision, tol in (("fp64", 2.6e-7), ("fp32c", 1e-6 * 2 * ds.bbox_radius(p))):
        gp, gn = _plugin(p, nr, r, precision).project_points(q)
        assert np.abs(gp - op)[keep].max(initial=0.0) <= tol
        assert np.array_equal(gp[-1], q[-1]) and not gn[-1].any()  # an empty ball: the query, no normal


@pytest.mark.parametrize("precision", ["fp32c", "fp64"])
def test_query_counts_give_the_same_bits(precision):
    p, nr = ds.torus(20000, seed=53)
    q = ds.jitter_queries(p[::7], 0.02, seed=54)
    ap = _plugin(p, nr, 0.15, precision)
    ref = ap.project_points(q, 2)
    for m in (1, 15, 16, 17, 31, 32, 33, 500):
        got = ap.project_points(q[:m], 2)
        assert np.array_equal(got[0], ref[0][:m]) and np.array_equal(got[1], ref[1][:m])


def test_many_points_in_one_leaf():
    p, nr = ds.sphere(2000, seed=55, noise=0.02)
    q = ds.jitter_queries(p[:40], 0.02, seed=56)
    a = _plugin(p, nr, 0.5, "fp64").project_points(q)
    b = _plugin(p, nr, 0.5, "fp64", maxNumberOfPointsPerLeaf=5000).project_points(q)  # one leaf, one range
    assert np.abs(a[0] - b[0]).max() <= 1.3e-7
