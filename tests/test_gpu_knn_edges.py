"""kNN APSS at the edges of the candidate arrays (8, 16, 32 and 64 slots), with clouds smaller than k,
exact ties in distance, and queries on points (distance 0)."""
import numpy as np
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds
from oracle import bind

pytestmark = pytest.mark.gpu


def _run(p, n, q, k, precision):
    R = ds.bbox_radius(p)
    sig = [0.2 * R, 0.4 * R]
    t = A.APSSOctree().build(p, n)
    t.knnMode(True, k)
    ap = A.Fastapss(t, A.Kernel(type=2, sigmas=sig))
    ap.set_precision(precision)
    ap.set_semantics("ref_cpu")
    got = ap.project_points(q)
    o = bind.OracleTree(p, n)
    ref = o.project(q, bind.make_kernel(type=2, sigmas=sig),
                    bind.make_params(cutoff=2.0, semantics="ref_cpu", mode="knn", knn=min(k, len(p))), precision=1)
    return got, ref, 2 * R


@pytest.mark.parametrize("k", [7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64])
@pytest.mark.parametrize("n", [40, 3000])
def test_knn_slots(k, n):
    p, nr = ds.sphere(n, seed=11, noise=0.05)
    q = np.concatenate([ds.jitter_queries(p[:300], 0.05, seed=12), p[:50]])  # the last 50 at distance 0
    (gp, gn), (op, on), diag = _run(p, nr, q, k, "fp64")
    # the FP64 form: the float32 rounding of positions below 2 (1.2e-7) over the diagonal
    assert np.abs(gp - op).max() <= 1.3e-7
    assert np.abs(gn - on).max() <= 1.3e-7


@pytest.mark.parametrize("k", [8, 20, 32])
def test_knn_ties(k):
    """Every point twice, half of them as a lattice: equal distances everywhere; the same pair of
    points comes with the same normal, so either of two tied twins gives the same sums."""
    p, nr = ds.sphere(1000, seed=13, noise=0.02)
    p2, n2 = np.repeat(p, 2, 0), np.repeat(nr, 2, 0)
    q = ds.jitter_queries(p[:200], 0.02, seed=14)
    (gp, _), (op, _), _ = _run(p2, n2, q, k, "fp64")
    assert np.abs(gp - op).max() <= 1.3e-7
