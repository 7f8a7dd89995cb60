"""The curve that queries are sorted along: a bijection whose consecutive cells share a face."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def curve(tmp_path_factory):
    d = tmp_path_factory.mktemp("curve")
    src, so = d / "c.cpp", d / "c.so"
    src.write_text('#include "%s"\n'
                   'extern "C" void keys(const unsigned* xyz, unsigned n, unsigned* out) {\n'
                   '  for (unsigned i = 0; i < n; ++i) out[i] = mlod::curve_key(xyz[3*i], xyz[3*i+1], xyz[3*i+2]);\n'
                   '}\n' % os.path.join(ROOT, "mlodsurfaces_amd", "csrc", "curve.h"))
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))

    def keys(xyz):
        a = np.ascontiguousarray(xyz, np.uint32)
        out = np.zeros(len(a), np.uint32)
        lib.keys(a.ctypes.data_as(ctypes.c_void_p), len(a), out.ctypes.data_as(ctypes.c_void_p))
        return out

    return keys


@pytest.mark.parametrize("bits", [1, 2, 5])
def test_coarse_cells_follow_the_curve(curve, bits):
    """The cells of a 2^bits grid (their first fine cell): all keys' leading bits, neighbours in turn."""
    n = 1 << bits
    g = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3)
    lead = curve(g << (10 - bits)) >> (3 * (10 - bits))
    assert np.array_equal(np.sort(lead), np.arange(n ** 3))
    path = g[np.argsort(lead)]
    assert np.all(np.abs(np.diff(path, axis=0)).sum(1) == 1)


def test_fine_cells_follow_the_curve(curve):
    """A block of the finest cells: distinct keys, and every key's successor in the block is next to it."""
    rng = np.random.default_rng(1)
    o = rng.integers(0, 1024 - 16, 3) // 16 * 16
    g = np.stack(np.meshgrid(*[np.arange(16)] * 3, indexing="ij"), -1).reshape(-1, 3) + o
    k = curve(g)
    s = np.argsort(k)
    assert np.array_equal(k[s] - k[s][0], np.arange(4096))
    assert np.all(np.abs(np.diff(g[s], axis=0)).sum(1) == 1)
