"""Low limits (loDistLimitSq, minDistSq) on the lane walks: where a leaf within the limit exists the answer is the
reference's first one in its own order, bit for bit that of the per-lane form.  Limits below, at and beyond the
distances (integer distances to the faces of a box meet the limit exactly), below and above the upper limit, and
limits per query."""
import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import synth

pytestmark = pytest.mark.gpu


def box(n):
    """the surface of [0, n]^3 in unit squares"""
    a, b = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    q = np.stack([a, b, a + 1, b, a + 1, b + 1, a, b + 1], -1).reshape(-1, 4, 2).astype(np.float32)
    quads = []
    for axis in range(3):
        for side in (0.0, float(n)):
            p = np.insert(q, axis, side, axis=2)
            quads.append(p if (axis == 1) != (side > 0) else p[:, ::-1])
    v = np.concatenate(quads).reshape(-1, 3)
    v, at = np.unique(v, axis=0, return_inverse=True)
    at = at.reshape(-1, 4)
    return v, np.concatenate([at[:, [0, 1, 2]], at[:, [0, 2, 3]]]).astype(np.int32)


def hills(n):
    rng = np.random.default_rng(1)
    x, y = np.meshgrid(np.arange(n, dtype=np.float32), np.arange(n, dtype=np.float32), indexing="ij")
    v = np.stack([x.ravel(), y.ravel(), rng.random(n * n).astype(np.float32)], 1)
    i, j = (k.ravel() for k in np.meshgrid(np.arange(n - 1), np.arange(n - 1), indexing="ij"))
    a = i * n + j
    return v, np.concatenate([np.stack([a, a + n, a + n + 1], 1), np.stack([a, a + n + 1, a + 1], 1)]).astype(np.int32)


MESHES = {"one": lambda: tuple(x[:k] for x, k in zip(synth.bumpy_icosphere(0, 1, 1), (12, 1))),
          "box": lambda: box(7), "bumpy": lambda: synth.bumpy_icosphere(4, 9, 3), "wide": lambda: hills(2060)}


@pytest.mark.parametrize("name", ["one", "box", "bumpy", "wide"])
@pytest.mark.parametrize("lo", [1e-12, 0.04, 1.0, 4.0, 1e9])
def test_low_limits_match_per_lane(name, lo):
    v, f = MESHES[name]()
    mesh = M.Mesh(v, f)
    proj, fwn = M.PointsToMeshProjector(), M.FastWindingNumber(mesh)
    proj.updateMeshData(mesh)
    rng = np.random.default_rng(5)
    low, high = v.min(0) - 2, v.max(0) + 2
    pts = np.concatenate([rng.uniform(low, high, (1500, 3)), np.round(rng.uniform(low, high, (1500, 3))),
                          v[rng.integers(0, len(v), 100)]]).astype(np.float32)
    dims = np.array([13, 11, 12], np.int32)
    step = np.maximum(1.0, np.round((high - low) / dims)).astype(np.float32)
    xf = np.concatenate([np.diag(step).ravel(), np.round(low)]).astype(np.float32)

    def answers():
        out = []
        for up in (M.FLT_MAX, 2.0, 0.5):
            out.append(proj.findProjections(pts, upDistLimitSq=up, loDistLimitSq=lo))
            for null in (True, False):
                o = M.DistanceToMeshOptions(minDistSq=lo, maxDistSq=up)
                o.nullOutsideMinMax = null
                out.append(fwn.calcFromGridWithDistances(dims, xf, o))
        return [np.ascontiguousarray(a).view(np.uint8) for a in out]

    got = answers()
    mesh.set_mode("traversal", "per_lane")
    for k, (a, b) in enumerate(zip(got, answers())):
        assert np.array_equal(a, b), k
