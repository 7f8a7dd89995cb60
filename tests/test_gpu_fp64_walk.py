"""The FP64 form's walk and weights against the FP64 oracle: whole exponents by products and the others by pow, one sigma
or an odd number of them, a sigma whose exponents leave the range of a whole number, min depths on both sides of the
tree's depth.  1e-7 of the diagonal: the outputs are float32, and their unit in the last place is the floor."""
import numpy as np
import pytest

from gpu_util import gpu_project, gpu_tree, rel_err
from mlodsurfaces_amd import datasets as ds

pytestmark = pytest.mark.gpu

KERNELS = [dict(type=1, exponent=float(e), constant_shift=c) for e in (1, 2, 3, 4, 5) for c in (0.0, 1e-3)] + [
    dict(type=1, exponent=2.5, constant_shift=1e-3), dict(type=0, sigma=0.06, constant_shift=1e-5),
    dict(type=2, sigmas=[0.06]), dict(type=2, sigmas=[0.03, 0.06, 0.12]),
    dict(type=2, sigmas=[1e-8, 0.04, 0.08, 0.16])]


@pytest.fixture(scope="module")
def scene(oracle_built):
    p, n = ds.torus(6000, seed=41)
    return p, n, gpu_tree(p, n), oracle_built.OracleTree(p, n), ds.jitter_queries(p[:333], 0.01, seed=42)


def _case(k):
    # w = (c' / d^2)^5 without a shift leaves the fit to one or two points: its FP64 sums cancel, in the oracle as on the
    # GPU (pow is called in both), and the two differ by up to 3e-7
    alone = pytest.mark.xfail(reason="the fit is ill-conditioned in FP64 itself", strict=False)
    return pytest.param(k, id="-".join(str(v) for v in k.values()),
                        marks=[alone] if k.get("exponent") == 5.0 and k["constant_shift"] == 0.0 else [])


@pytest.mark.parametrize("kernel", [_case(k) for k in KERNELS])
@pytest.mark.parametrize("semantics,min_depth", [("ref_gpu", 0), ("ref_cpu", 0), ("ref_gpu", 2), ("ref_gpu", 12)])
def test_fp64_walk(oracle_built, scene, kernel, semantics, min_depth):
    p, n, tree, o, q = scene
    print("case", kernel, semantics, min_depth, flush=True)
    got, _, _ = gpu_project(tree, q, kernel, cutoff=2.0, min_depth=min_depth, semantics=semantics, precision="fp64")
    ref, _ = o.project(q, oracle_built.make_kernel(**kernel),
                       oracle_built.make_params(cutoff=2.0, min_depth=min_depth, semantics=semantics), precision=1)
    assert rel_err(got, ref.astype(np.float32), 2 * ds.bbox_radius(p)).max() < 1e-7
