"""Square roots and quotients of winding numbers: the short sequences that the kernels use inside [2^-60, 2^60) give the
correctly rounded results.  Roots: every float of the range.  Quotients num / (sqrt(dd) dd): that they scale exactly with dd
is checked for every float; of the 2^24 mantissas that are left for dd, a spread of 2^18 with every mantissa of num (all of
them take a minute)."""
import ctypes
import os

import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import build, synth

pytestmark = pytest.mark.gpu


def lib():
    if not os.path.exists(build.MID_MATH_LIB):
        build.build_mid_math()
    M.lib()      # the HIP runtime that the library uses comes first
    so = ctypes.CDLL(build.MID_MATH_LIB)
    for f in (so.mid_roots, so.mid_scales, so.mid_quotients):
        f.restype = ctypes.c_longlong
    so.mid_quotients.argtypes = [ctypes.c_uint32] * 3
    return so


def test_roots_are_correctly_rounded():
    assert lib().mid_roots() == 0


def test_results_scale_with_powers_of_four():
    assert lib().mid_scales() == 0


# an odd stride visits different mantissas throughout [1, 4)
@pytest.mark.parametrize("first", range(4))
def test_quotients_are_correctly_rounded(first):
    assert lib().mid_quotients(first, 1 << 16, 4 * 16411 + 1) == 0


@pytest.mark.parametrize("level", [0, 2, 5])
def test_wave_form_has_the_per_lane_form_s_bits(level):
    """The walk per wave and the walk per lane visit the same records in the same order with the same operations."""
    v, f = synth.bumpy_icosphere(level, 8, 3)
    mesh = M.Mesh(v, f)
    fwn = M.FastWindingNumber(mesh)
    pts = synth.projection_queries(v, f, 5003, 4)
    dims, xf, _ = synth.grid_for_mesh(v, (19, 16, 13))

    def answers():
        return fwn.calcFromVector(pts, 2.0).view(np.uint32), fwn.calcFromGrid(dims, xf, 2.0).view(np.uint32)

    got = answers()
    mesh.set_mode("traversal", "per_lane")
    for g, w in zip(got, answers()):
        assert np.array_equal(g, w)


def test_wave_form_has_the_per_lane_form_s_bits_above_2_23_faces():
    """The same where the records are addressed by number instead of by byte offset."""
    n = 2060
    rng = np.random.default_rng(4)
    x, y = np.meshgrid(np.arange(n, dtype=np.float32), np.arange(n, dtype=np.float32), indexing="ij")
    v = np.stack([x.ravel(), y.ravel(), rng.random(n * n).astype(np.float32)], 1)
    i, j = (k.ravel() for k in np.meshgrid(np.arange(n - 1), np.arange(n - 1), indexing="ij"))
    a = i * n + j
    f = np.concatenate([np.stack([a, a + n, a + n + 1], 1), np.stack([a, a + n + 1, a + 1], 1)]).astype(np.int32)
    assert len(f) > 1 << 23
    mesh = M.Mesh(v, f)
    fwn = M.FastWindingNumber(mesh)
    pts = (rng.random((2000, 3)) * [n, n, 6] - [0, 0, 3]).astype(np.float32)
    dims, xf, _ = synth.grid_for_mesh(v, (9, 8, 5))
    got = fwn.calcFromVector(pts, 2.0), fwn.calcFromGrid(dims, xf, 2.0)
    mesh.set_mode("traversal", "per_lane")
    want = fwn.calcFromVector(pts, 2.0), fwn.calcFromGrid(dims, xf, 2.0)
    for g, w in zip(got, want):
        assert np.array_equal(g.view(np.uint32), w.view(np.uint32))
