"""The FP32 forms' walks, one lane a query with node records staged through LDS and, for small batches, eight lanes a
query: the same bits from both, ragged query counts (lanes without a query beside lanes that have one), multi-point
leaves, trees of one leaf and of one level, min depths on both sides of the tree's depth, and a tree of 2^26 nodes
or more (64-bit record offsets)."""
import numpy as np
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds
from oracle import bind

pytestmark = pytest.mark.gpu


def _plugin(t, sig, precision, cutoff=2.0, min_depth=0, semantics="ref_gpu"):
    ap = A.Fastapss(t, A.Kernel(type=2, sigmas=sig))
    ap.setScalingProtectionSphere(cutoff)
    ap.setMinDepth(min_depth)
    ap.set_precision(precision)
    ap.set_semantics(semantics)
    return ap


@pytest.fixture(scope="module")
def cloud():
    p, n = ds.torus(20000, seed=21)
    R = ds.bbox_radius(p)
    return p, n, [0.02 * R, 0.04 * R, 0.08 * R, 0.16 * R], 2 * R


@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 127, 129, 257])
@pytest.mark.parametrize("precision", ["fp32", "fp32c"])
def test_ragged_counts_give_the_same_bits(cloud, m, precision):
    p, n, sig, _ = cloud
    t = A.APSSOctree().build(p, n)
    q = ds.jitter_queries(p[:300], 0.02, seed=22)
    ap = _plugin(t, sig, precision)
    ref = ap.project_points(q, 2)
    got = ap.project_points(q[:m], 2)
    assert np.array_equal(got[0], ref[0][:m]) and np.array_equal(got[1], ref[1][:m])


@pytest.mark.parametrize("max_depth,leaf,min_depth", [(1, 1, 0), (2, 1, 1), (4, 1, 0), (5, 1, 13), (12, 7, 0), (12, 1, 20),
                                                      (12, 30000, 0), (12, 1, 1)])
@pytest.mark.parametrize("semantics", ["ref_gpu", "ref_cpu"])
def test_leaf_and_level_edges(cloud, max_depth, leaf, min_depth, semantics):
    p, n, sig, diag = cloud
    t = A.APSSOctree().build(p, n, maxDepth=max_depth, maxNumberOfPointsPerLeaf=leaf)
    q = ds.jitter_queries(p[:200], 0.02, seed=23)
    out = {f: _plugin(t, sig, f, 2.0, min_depth, semantics).project_points(q, 1)[0] for f in ("fp64", "fp32c")}
    # REF_CPU keeps one point of a leaf: a one-leaf tree then has no sphere, in any form
    if not (semantics == "ref_cpu" and (leaf > len(p) or max_depth <= 2)):
        assert np.abs(out["fp32c"] - out["fp64"]).max() <= 1e-6 * diag  # the compensated form's budget
    else:
        assert out["fp32c"].shape == out["fp64"].shape


KERNELS = {"mg": dict(type=2, sigmas=[0.03, 0.06, 0.12]), "mg11": dict(type=2, sigmas=[0.02 * 1.3 ** i for i in range(11)]),
           "rat": dict(type=1, exponent=4.0, constant_shift=1e-3), "gauss": dict(type=0, sigma=0.1)}


@pytest.mark.parametrize("kernel", sorted(KERNELS))
@pytest.mark.parametrize("precision", ["fp32", "fp32c"])
@pytest.mark.parametrize("semantics", ["ref_gpu", "ref_cpu"])
@pytest.mark.parametrize("max_depth,leaf,min_depth,cutoff", [(12, 1, 0, 2.0), (5, 1, 0, 1.4), (12, 9, 1, 3.0), (3, 1, 2, 2.0)])
def test_lane_and_group_walks_give_the_same_bits(cloud, kernel, precision, semantics, max_depth, leaf, min_depth, cutoff):
    """60000 queries take a lane each, 999 of them a group of eight; some lie beyond every cutoff."""
    p, n, _, _ = cloud
    t = A.APSSOctree().build(p, n, maxDepth=max_depth, maxNumberOfPointsPerLeaf=leaf)
    q = ds.jitter_queries(np.tile(p, (3, 1)), 0.03, seed=24)
    q[::100] *= 4.0
    ap = A.Fastapss(t, A.Kernel(**KERNELS[kernel]))
    ap.setScalingProtectionSphere(cutoff)
    ap.setMinDepth(min_depth)
    ap.set_precision(precision)
    ap.set_semantics(semantics)
    ref = ap.project_points(q, 2)
    got = ap.project_points(q[:999], 2)
    for g, r in zip(got, ref):
        assert np.array_equal(g.view(np.int32), r[:999].view(np.int32))


def test_records_beyond_32_bit_offsets():
    """18M pairs of near points: a chain of nodes for each pair, so the tree has more than 2^26 nodes."""
    rng = np.random.default_rng(31)
    k = 18_000_000
    u = rng.standard_normal((k, 3), dtype=np.float32)
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    c = u * (1.0 + 0.25 * rng.random((k, 1), dtype=np.float32))
    p = np.concatenate([c, c + np.float32(2e-4) * rng.standard_normal((k, 3), dtype=np.float32)])
    n = np.concatenate([u, u])
    t = A.APSSOctree().build(p, n)
    assert t.info()["n_nodes"] >= 1 << 26
    sig = [0.1, 0.2]
    q = p[rng.integers(0, len(p), 2000)] + rng.uniform(-0.02, 0.02, (2000, 3)).astype(np.float32)
    out = {f: _plugin(t, sig, f).project_points(q, 1)[0] for f in ("fp64", "fp32c", "fp32")}
    diag = 2 * t.radius()
    assert np.abs(out["fp32c"] - out["fp64"]).max() <= 1e-6 * diag
    assert np.abs(out["fp32"] - out["fp64"]).max() <= 1e-5 * diag
    many = np.tile(q, (26, 1))  # a lane a query
    assert np.array_equal(_plugin(t, sig, "fp32c").project_points(many, 1)[0][:2000], out["fp32c"])


@pytest.mark.parametrize("k", [-16, 16])
@pytest.mark.parametrize("m", [999, 60000])
def test_plain_form_scales_exactly(cloud, k, m):
    """A cloud scaled by a power of two goes through the same roundings: its walk's quotients by the nodes' areas,
    blend ratios and square roots are right at every exponent, so the results scale to the bit."""
    p, n, sig, _ = cloud
    s = np.float32(2.0) ** k
    q = ds.jitter_queries(np.tile(p, (3, 1)), 0.02, seed=25)[:m]
    got = [_plugin(A.APSSOctree().build(p * f, n), [float(np.float32(x) * f) for x in sig], "fp32").project_points(q * f, 2)
           for f in (np.float32(1.0), s)]
    assert np.array_equal(got[0][0] * s, got[1][0]) and np.array_equal(got[0][1], got[1][1])
