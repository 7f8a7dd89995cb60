"""Global APSS on the matrix cores: point counts at the edges of a tile and a round, query counts at the edges of
a workgroup and on both sides of the split's limit, against the FP64 oracle."""
import numpy as np
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds
from oracle import bind

pytestmark = pytest.mark.gpu

KERNELS = {"mg": dict(type=2, sigmas=[0.3, 0.6, 1.2]), "rat": dict(type=1, exponent=4.0, constant_shift=1e-3),
           "gauss": dict(type=0, sigma=0.4)}


def _project(p, n, q, kernel, precision, steps=1):
    t = A.APSSOctree().build(p, n)
    ap = A.GlobalAPSS(t, A.Kernel(**KERNELS[kernel]))
    ap.set_precision(precision)
    ap.set_semantics("ref_cpu")
    return ap.project_points(q, steps)


@pytest.mark.parametrize("n", [8, 63, 64, 65, 255, 256, 257, 513, 1500])
@pytest.mark.parametrize("kernel", sorted(KERNELS))
def test_point_counts(n, kernel):
    p, nr = ds.sphere(n, seed=41, noise=0.02)
    q = ds.jitter_queries(np.repeat(p[:8], 5, 0), 0.1, seed=42)
    o = bind.OracleTree(p, nr)
    op, on = o.project(q, bind.make_kernel(**KERNELS[kernel]), bind.make_params(cutoff=2.0, semantics="ref_cpu", mode="global"),
                       precision=1)
    diag = 2 * ds.bbox_radius(p)
    gp, gn = _project(p, nr, q, kernel, "fp64")
    assert np.abs(gp - op).max() <= 1.3e-7 * 2  # the float32 rounding of positions below 2
    gp, gn = _project(p, nr, q, kernel, "fp32c")
    assert np.abs(gp - op).max() <= 1e-6 * diag


@pytest.mark.parametrize("precision", ["fp32c", "fp64"])
def test_query_counts_and_splits_give_the_same_bits(precision):
    p, nr = ds.torus(700, seed=43)
    q = ds.jitter_queries(np.tile(p, (13, 1)), 0.05, seed=44)
    ref = _project(p, nr, q, "mg", precision, 2)  # 9100 queries: four wavefronts a workgroup
    assert len(q) > 16 * 512
    for m in (1, 15, 16, 17, 500, 8176):  # sixteen
        got = _project(p, nr, q[:m], "mg", precision, 2)
        assert np.array_equal(got[0], ref[0][:m]) and np.array_equal(got[1], ref[1][:m])
