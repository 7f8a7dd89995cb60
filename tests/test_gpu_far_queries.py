"""Queries far beyond the cloud (sentinels of 1e19 to FLT_MAX among them), where squared distances leave the float range
and every Gaussian underflows: the weights are then the kernel's constant shift, and the step goes towards the sphere of
the whole cloud."""
import numpy as np
import pytest

from gpu_util import gpu_project, gpu_tree
from mlodsurfaces_amd import datasets as ds

pytestmark = pytest.mark.gpu

FM = np.finfo(np.float32).max
FAR = np.array([[FM, FM, FM], [-FM, 0, 0], [0, FM, 0], [1e20, 0, 1e20], [1e19, 1e19, 0], [0, 1e17, 0], [1e12, 0, 2e12],
                [100, 200, 50]], np.float32)


@pytest.fixture(scope="module")
def scene(oracle_built):
    p, n = ds.torus(5000, seed=71)
    return gpu_tree(p, n), oracle_built.OracleTree(p, n)


@pytest.mark.parametrize("mode", ["mlod", "global"])
@pytest.mark.parametrize("min_depth", [0, 2])
@pytest.mark.parametrize("sigmas", [1, 2, 3, 5, 9, 10, 11, 30])
def test_fp64_form(oracle_built, scene, sigmas, min_depth, mode):
    tree, o = scene
    k = dict(type=2, sigmas=[0.05 * 1.1 ** i for i in range(sigmas)], constant_shift=1e-3)
    kw = dict(cutoff=2.0, min_depth=min_depth, semantics="ref_cpu" if mode == "global" else "ref_gpu", mode=mode)
    got, nrm, _ = gpu_project(tree, FAR, k, precision="fp64", **kw)
    ref, rn = o.project(FAR, oracle_built.make_kernel(**k), oracle_built.make_params(**kw), precision=1)
    assert np.linalg.norm(rn, axis=1).min() > 0.99  # the definition gives every one of them a normal
    scale = np.abs(FAR).max(1, keepdims=True).astype(np.float64)
    assert (np.abs(got - ref) / scale).max() <= 2.4e-7  # a float32 unit in the last place or two of the largest coordinate
    assert np.abs(nrm - rn).max() <= 2.4e-7


@pytest.mark.parametrize("mode,m", [("mlod", 5), ("mlod", 60000), ("knn", 5), ("global", 5)])  # (a batch of 5: eight lanes each)
@pytest.mark.parametrize("precision", ["fp32", "fp32c"])
def test_float_forms_take_any_number_of_sigmas(scene, precision, mode, m):
    """The five farthest: every float squared distance overflows, the weights are the shift whatever the sigmas."""
    tree, _ = scene
    q = np.tile(FAR[:5], (m // 5, 1))
    out = {}
    for sigmas in (2, 1, 3, 5, 7, 8, 9, 10, 11, 12, 30, 32):
        k = dict(type=2, sigmas=[0.05 * 1.1 ** i for i in range(sigmas)], constant_shift=1e-3)
        out[sigmas] = gpu_project(tree, q, k, cutoff=2.0, semantics="ref_gpu" if mode == "mlod" else "ref_cpu",
                                  precision=precision, mode=mode)[:2]
    for sigmas, o in out.items():
        for a, b in zip(o, out[2]):
            assert np.array_equal(a.view(np.int32), b.view(np.int32)), sigmas
    if precision == "fp32" and mode != "knn":  # (the other form's offsets overflow too, and knn's distances)
        assert np.linalg.norm(out[2][1], axis=1).min() > 0.99


@pytest.mark.parametrize("semantics", ["ref_gpu", "ref_cpu"])
@pytest.mark.parametrize("precision", ["fp32", "fp32c"])
@pytest.mark.parametrize("min_depth", [1, 2, 13])
@pytest.mark.parametrize("scale", [0, -62])  # at -62 the nodes' areas are subnormal: their reciprocals overflow
def test_no_blending_above_the_min_depth(scale, min_depth, precision, semantics):
    """Infinite distances, and areas without a reciprocal, against the wave walk, which keeps such nodes' factors apart."""
    s = np.float32(2.0) ** scale
    p, n = ds.torus(5000, seed=71)
    tree = gpu_tree(p * s, n)
    q = np.concatenate([FAR, ds.jitter_queries(p[:20], 0.02, seed=72) * s])
    kw = dict(kernel=dict(type=0, sigma=float(0.05 * s), constant_shift=1e-3), min_depth=min_depth, semantics=semantics,
              precision=precision)
    ref = gpu_project(tree, q, traversal="wave", **kw)[:2]
    for m in (1, 2000):  # eight lanes a query; one
        got = gpu_project(tree, np.tile(q, (m, 1)), **kw)[:2]
        # the two walks add the same terms in the same order, but may fuse a multiply-add differently
        assert np.abs(got[1][:len(q)] - ref[1]).max() <= 1e-4
        assert (np.abs(got[0][:len(q)].astype(np.float64) - ref[0]) / np.abs(q).max(1, keepdims=True)).max() <= 1e-6


@pytest.mark.parametrize("exponent", [1.0, 4.0, 2.5])
@pytest.mark.parametrize("precision", ["fp32", "fp32c"])
def test_rational_weights_near_the_end_of_the_float_range(precision, exponent):
    """Squared distances between 2^126 and 2^128, whose reciprocals are subnormal: a large cloud (2^58 across) with a
    shift of its scale, the nearest points of queries 1.1e19 to 1.7e19 away: weights and a fit as in the FP64 form."""
    s = np.float32(2.0) ** 58
    p, n = ds.torus(3000, seed=73)
    p = p * s
    shift = float(np.float32(8e31))
    u = np.random.default_rng(74).standard_normal((16, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    q = (u * np.linspace(1.1e19, 1.7e19, 16)[:, None]).astype(np.float32)
    got, _, _ = gpu_project(gpu_tree(p, n), q, dict(type=1, exponent=exponent, constant_shift=shift), mode="knn", knn=20,
                            precision="fp64")
    out, nrm, _ = gpu_project(gpu_tree(p, n), q, dict(type=1, exponent=exponent, constant_shift=shift), mode="knn", knn=20,
                              precision=precision)
    assert np.isfinite(got).all() and np.isfinite(out).all() and np.linalg.norm(nrm, axis=1).min() > 0.99
