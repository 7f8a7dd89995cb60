"""The FP64 form with w = (c' / d^2)^5 and no shift, a kernel that leaves the fit to one or two points: the sums cancel in
FP64 itself, so the bound is that of the queries where they do not, and a wider one for all."""
import numpy as np
import pytest

from gpu_util import gpu_project, gpu_tree, rel_err
from mlodsurfaces_amd import datasets as ds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("semantics,min_depth", [("ref_gpu", 0), ("ref_cpu", 0), ("ref_gpu", 2), ("ref_gpu", 12)])
def test_fifth_power(oracle_built, semantics, min_depth):
    p, n = ds.torus(6000, seed=41)
    k = dict(type=1, exponent=5.0, constant_shift=0.0)
    q = ds.jitter_queries(p[:333], 0.01, seed=42)
    got, _, _ = gpu_project(gpu_tree(p, n), q, k, cutoff=2.0, min_depth=min_depth, semantics=semantics, precision="fp64")
    o = oracle_built.OracleTree(p, n)
    par = oracle_built.make_params(cutoff=2.0, min_depth=min_depth, semantics=semantics)
    ref, _ = o.project(q, oracle_built.make_kernel(**k), par, precision=1)
    err = rel_err(got, ref.astype(np.float32), 2 * ds.bbox_radius(p))
    S = o.stats(q, oracle_built.make_kernel(**k), par)
    spread = S[:, 8] / S[:, 0] - (S[:, 1:4] ** 2).sum(1) / S[:, 0] ** 2  # of the weighted points, out of sums of order 1
    clear = spread > 1e-7  # 1e-16 / spread below 1e-9
    assert clear.sum() > 100
    assert err[clear].max() < 1e-7
    assert err.max() < 1e-6
