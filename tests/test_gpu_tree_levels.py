"""The GPU tree build at the sizes and ties where its two phases can go wrong: around the largest subtree that
one block builds (1024 leaves) and the chunk of a level kernel (4096), and pivots that share their first, their
first two and all three keys with other leaves (rows of a planar grid, stacked copies of one grid, copies of one
triangle).  Nodes and dipoles equal the host build bit for bit."""
import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import synth

pytestmark = pytest.mark.gpu


def _grid(g, copies):
    x, y = np.meshgrid(np.arange(g + 1, dtype=np.float32), np.arange(g + 1, dtype=np.float32))
    v = np.stack([x.ravel(), y.ravel(), np.zeros(x.size, np.float32)], 1)
    i, j = (k.ravel() for k in np.meshgrid(np.arange(g), np.arange(g)))
    a = i * (g + 1) + j
    f = np.concatenate([np.stack([a, a + 1, a + g + 2], 1), np.stack([a, a + g + 2, a + g + 1], 1)])
    return v, np.concatenate([f] * copies).astype(np.int32)


def _cases():
    v, f = synth.bumpy_icosphere(5, 8, 3)
    rng = np.random.default_rng(2)
    f = f[rng.permutation(len(f))]
    for n in (3, 1023, 1024, 1025, 2047, 2049, 4097, 8193, 20480):
        yield f"sphere-{n}", v, f[:n]
    yield ("grid-200",) + _grid(200, 1)
    yield ("grid-40-x7",) + _grid(40, 7)
    yield "one-triangle-x5000", v[:3], np.tile(np.array([[0, 1, 2]], np.int32), (5000, 1))
    w, g = _grid(70, 1)
    yield "grid-z-steps", (w + np.c_[np.zeros((len(w), 2)), rng.integers(0, 3, len(w))]).astype(np.float32), g


@pytest.mark.parametrize("case", list(_cases()), ids=lambda c: c[0])
def test_tree_equals_host_build(case):
    name, v, f = case
    gm = M.Mesh(v, f)
    nodes, dips = gm.tree()
    hn, hd, depth = M.build_tree_host(v, f)
    assert gm.depth() == depth
    assert np.array_equal(nodes.view(np.uint8), hn.view(np.uint8))
    assert np.array_equal(dips.view(np.uint8), hd.view(np.uint8))
