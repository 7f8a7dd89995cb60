"""Point areas below the normal floats: a root box far smaller than the cloud (the build keeps the box it is given) makes
every leaf's diagonal, whose square over its points is their area, as small as one likes.  The plain form is then as
close to the FP64 form as it is with normal areas, up to the few bits that such areas and their moments have."""
import numpy as np
import pytest

from gpu_util import gpu_project
from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds

pytestmark = pytest.mark.gpu

KERNELS = {"mg": dict(type=2, sigmas=[0.2, 0.4, 0.8]), "rat": dict(type=1, exponent=2.0, constant_shift=0.05)}


def _errors(box, kernel, mode, traversal, m, reach):
    p, n = ds.torus(1500, seed=81)
    t = A.APSSOctree()
    t.setRootBoundingBox([0, 0, 0], [2.0 ** box] * 3)
    t.build(p, n, updateRootBoundingBox=False)
    a = t.dump()["areas"].min()
    assert 0 < a and (a < 2.0 ** -126) == (box < -46)
    q = np.tile(ds.jitter_queries(p[::10], 0.05, seed=82), (m, 1))
    # cutoffs in box edges: the walk is the same in every box, and so is the step bound
    kw = dict(cutoff=2.0 ** (reach - box), semantics="ref_gpu" if mode == "mlod" else "ref_cpu", mode=mode, traversal=traversal,
              step_max=10.0)
    ref, rn, _ = gpu_project(t, q, KERNELS[kernel], precision="fp64", **kw)
    got, gn, _ = gpu_project(t, q, KERNELS[kernel], precision="fp32", **kw)
    assert np.linalg.norm(rn, axis=1).min() > 0.99
    return a, np.abs(got - ref).max(), np.abs(gn - rn).max()


@pytest.mark.parametrize("kernel", sorted(KERNELS))
@pytest.mark.parametrize("mode,traversal,m", [("global", "lane", 1), ("mlod", "lane", 1), ("mlod", "lane", 400), ("mlod", "wave", 1)])
@pytest.mark.parametrize("box", [-50, -54])
@pytest.mark.parametrize("reach", [3, 14])  # far nodes at several levels; leaves of many points
def test_plain_form(kernel, mode, traversal, m, box, reach):
    _, p0, n0 = _errors(-46, kernel, mode, traversal, m, reach)
    a, ep, en = _errors(box, kernel, mode, traversal, m, reach)
    # the moments a p, a p.p of such areas are off by 2^-150 / a, the fit's outputs by a hundredfold of that
    assert ep <= 2 * p0 + 100 * 2.0 ** -150 / a and en <= 2 * n0 + 100 * 2.0 ** -150 / a
