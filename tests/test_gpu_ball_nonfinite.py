"""Ball APSS with points whose normal or position is not finite (the build takes them as they are): they count for the
queries whose ball holds them and for no other."""
import numpy as np
import pytest

from mlodsurfaces_amd import apss as A
from mlodsurfaces_amd import datasets as ds

pytestmark = pytest.mark.gpu

R = 0.15


def _plugin(p, n, kernel, precision):
    t = A.APSSOctree().build(p, n)
    t.ballMode(True, R)
    ap = A.Fastapss(t, A.Kernel(**kernel))
    ap.set_precision(precision)
    ap.set_semantics("ref_cpu")
    return ap


KERNELS = {"mg": dict(type=2, sigmas=[0.05, 0.1, 0.2]), "rat": dict(type=1, exponent=4.0, constant_shift=1e-3)}


@pytest.mark.parametrize("precision", ["fp32c", "fp64"])
@pytest.mark.parametrize("kernel", sorted(KERNELS))
@pytest.mark.parametrize("what,value", [("normal", np.nan), ("normal", np.inf), ("normal", -np.inf), ("position", np.nan),
                                        ("position", np.inf)])
def test_only_the_balls_that_hold_the_point(precision, kernel, what, value):
    p, n = ds.torus(8000, seed=61)
    bad = [7, 8, 1000, 4000]
    pb, nb = p.copy(), n.copy()
    (nb if what == "normal" else pb)[bad, 1] = value
    q = np.concatenate([ds.jitter_queries(p[::17], 0.02, seed=62), ds.jitter_queries(p[bad], 0.02, seed=63)])
    ap = _plugin(pb, nb, KERNELS[kernel], precision)
    got = ap.project_points(q)
    d = np.linalg.norm(q[:, None].astype(np.float64) - p[bad][None], axis=2)
    assert not ((d > R * 0.999) & (d < R * 1.001)).any()
    holds = (d <= R).any(1) if what == "normal" else np.zeros(len(q), bool)  # (no ball reaches such a position)
    assert what == "position" or 10 < holds.sum() < len(q) // 2
    # a ball without the point: as in the cloud with the point out of reach (the tree's ranges may differ: the last bit)
    far_p, far_n = np.delete(p, bad, 0), np.delete(n, bad, 0)
    ref = _plugin(far_p, far_n, KERNELS[kernel], precision).project_points(q)
    tol = 2.4e-7  # a unit in the last place of float32 values below 2, either way
    for g, r in zip(got, ref):
        assert np.isfinite(g[~holds]).all()
        assert np.abs(g - r)[~holds].max() <= tol
    # a ball with it: no position (kept NaN, with a zero normal)
    if holds.any():
        assert not np.isfinite(got[0][holds]).all(1).any() and not got[1][holds].any()
    # and the same bits whichever queries share its wavefront
    for i in np.linspace(0, len(q) - 1, 23).astype(int):
        one = ap.project_points(q[i:i + 1])
        assert np.array_equal(one[0], got[0][i:i + 1], equal_nan=True) and np.array_equal(one[1], got[1][i:i + 1])
