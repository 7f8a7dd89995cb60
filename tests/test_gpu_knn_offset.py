"""kNN far from the origin and in root boxes much larger than the cloud, where cells' bounds round: every neighbour is
found (the k nearest of the float32 distances, by brute force; queries with a tie at the last one are left out)."""
import numpy as np
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds
from oracle import bind

pytestmark = pytest.mark.gpu

SIG = [0.1, 0.2]


@pytest.mark.parametrize("k", [8, 20])
@pytest.mark.parametrize("offset", [0.0, 100.0, 1000.0])
@pytest.mark.parametrize("box", [None, 1000.0])
def test_every_neighbour_is_found(box, offset, k):
    o = np.float32([offset, -offset, offset / 4])
    p, n = ds.torus(4000, seed=111)
    p, q = (p + o).astype(np.float32), (ds.jitter_queries(p[:400], 0.02, seed=112) + o).astype(np.float32)
    d = p[None] - q[:, None]
    d2 = np.sort((d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2], axis=1)  # in float32
    clear = d2[:, k - 1] < d2[:, k]
    assert clear.sum() > 150
    rb = None if box is None else [*(o - box), *(o + box)]
    t = A.APSSOctree()
    if rb is not None:
        t.setRootBoundingBox(rb[:3], rb[3:])
    t.build(p, n, updateRootBoundingBox=rb is None)
    t.knnMode(True, k)
    ap = A.Fastapss(t, A.Kernel(type=2, sigmas=SIG))
    ap.set_semantics("ref_cpu")
    ap.set_precision("fp64")
    gp, gn = ap.project_points(q)
    # the definition with those neighbours, sums about the query in FP64 (the FP64 form's own are global: 1e-16 |q|^2)
    x = p.astype(np.float64)[None] - q.astype(np.float64)[:, None]
    near = np.argsort((d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2], axis=1, kind="stable")[:, :k]
    x, nn = np.take_along_axis(x, near[..., None], 1), n.astype(np.float64)[near]
    e2 = (x * x).sum(2)
    w = sum(np.exp(-e2 / (2 * float(np.float32(s)) ** 2)) / float(np.float32(s)) ** 3 for s in SIG)
    sw, sp, sn = w.sum(1), (w[..., None] * x).sum(1), (w[..., None] * nn).sum(1)
    u4 = 0.5 * ((w * (x * nn).sum(2)).sum(1) - (sp * sn).sum(1) / sw) / ((w * e2).sum(1) - (sp * sp).sum(1) / sw)
    u = (sn - 2 * u4[:, None] * sp) / sw[:, None]
    u0 = -((sp * u).sum(1) + u4 * (w * e2).sum(1)) / sw
    un = np.linalg.norm(u, axis=1)
    s = (-2 * u0 / (un + np.sqrt(np.maximum(un * un - 4 * u4 * u0, 0))) / un)[:, None] * u
    nr = u + 2 * u4[:, None] * s
    nr /= np.linalg.norm(nr, axis=1, keepdims=True)
    # a wrong neighbour moves a normal by 1e-3 and more; the global sums by 1e-16 |q|^2 / (spacing of 0.03)^2, a hundredfold
    tol = 3e-7 + 1e-14 * float((o.astype(np.float64) ** 2).sum()) / 0.03 ** 2
    assert np.abs(gn - nr)[clear].max() <= tol
    assert np.abs(gp - (q.astype(np.float64) + s))[clear].max() <= tol + (offset + 2) * 2.0 ** -24
