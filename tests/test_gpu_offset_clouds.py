"""The compensated form far from the origin: its fit is in the query's frame, so a cloud moved by an exact offset has the
normals it had in the modes that sum points (a node's mean in the MLoD mode is rounded to float32 where it lies).
Coordinates on a grid of 2^-10, which floats hold up to 2^14; the same root box, moved, with cells on the grid."""
import numpy as np
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds
from oracle import bind

pytestmark = pytest.mark.gpu

KERNELS = {"mg": dict(type=2, sigmas=[0.05, 0.08, 0.128]), "rat": dict(type=1, exponent=4.0, constant_shift=1e-3)}


def _grid(x):
    return (np.round(np.asarray(x, np.float64) * 1024) / 1024).astype(np.float32)


@pytest.mark.parametrize("kernel", sorted(KERNELS))
@pytest.mark.parametrize("mode", ["ball", "global", "knn"])
@pytest.mark.parametrize("offset", [0.0, 64.0, 8192.0])
def test_normals_do_not_depend_on_the_offset(offset, mode, kernel):
    p, n = ds.torus(6000, seed=91)
    p, q = _grid(p), _grid(ds.jitter_queries(p[:300], 0.03, seed=92))
    o = bind.OracleTree(p, n, max_depth=8, root_box=[-2, -2, -2, 2, 2, 2])
    op, on = o.project(q, bind.make_kernel(**KERNELS[kernel]),
                       bind.make_params(cutoff=2.0, semantics="ref_cpu", mode=mode, ball_radius=0.15, knn=30), precision=1)
    f = np.float32(offset)
    t = A.APSSOctree()
    t.setRootBoundingBox([offset - 2] * 3, [offset + 2] * 3)
    t.build(p + f, n, updateRootBoundingBox=False, maxDepth=8)
    t.ballMode(mode == "ball", 0.15)
    t.knnMode(mode == "knn", 30)
    ap = (A.GlobalAPSS if mode == "global" else A.Fastapss)(t, A.Kernel(**KERNELS[kernel]))
    ap.set_precision("fp32c")
    ap.set_semantics("ref_cpu")
    gp, gn = ap.project_points(q + f)
    # float32 weights and offsets (3e-8 each) through the fit of a rational kernel, tenfold; the outputs' own rounding
    assert np.abs(gn - on).max() <= 1e-6
    assert np.abs(gp - f - op).max() <= 1e-6 + offset * 2.0 ** -24
