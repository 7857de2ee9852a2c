"""The lane walks (the default form of projections without a low limit and of signed distances without a
band) where they can go wrong: trees of a few leaves, waves with idle lanes, more leaves tying at one
distance than a lane's tie list holds, slivers, coplanar and duplicated faces, shapes far from the origin and
at extreme scales, limits that cut some queries off.  Records and distances are the oracle's bit for bit."""
import sys

import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _fan(n):
    """n triangles around one apex above a ring: the apex ties between all of them."""
    a = np.arange(n) * (2 * np.pi / n)
    v = np.concatenate([[[0, 0, 1.0]], np.stack([np.cos(a), np.sin(a), np.zeros(n)], 1)])
    i = np.arange(n)
    return v.astype(np.float32), np.stack([np.zeros(n, int), 1 + i, 1 + (i + 1) % n], 1).astype(np.int32)


def _plane(n):
    x, y = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
    v = np.stack([x, y, 0 * x], -1).reshape(-1, 3).astype(np.float32)
    i, j = (k.reshape(-1) for k in np.meshgrid(np.arange(n), np.arange(n), indexing="ij"))
    a = i * (n + 1) + j
    return v, np.concatenate([np.stack([a, a + n + 1, a + n + 2], 1), np.stack([a, a + n + 2, a + 1], 1)]).astype(np.int32)


def _tube(n, length):
    a = np.arange(n) * (2 * np.pi / n)
    ring = np.stack([np.cos(a), np.sin(a)], 1)
    v = np.concatenate([np.c_[ring, np.full(n, -length)], np.c_[ring, np.full(n, length)]]).astype(np.float32)
    i, j = np.arange(n), (np.arange(n) + 1) % n
    return v, np.concatenate([np.stack([i, j, j + n], 1), np.stack([i, j + n, i + n], 1)]).astype(np.int32)


def _mesh(name):
    if name.startswith("faces"):
        v, f = synth.bumpy_icosphere(2, 3, 7)
        return v, f[:int(name[5:])]
    if name == "fan":
        return _fan(203)
    if name == "plane":
        return _plane(13)
    if name == "tube":
        return _tube(333, 40.0)
    v, f = synth.bumpy_icosphere(3, 5, 2)
    if name == "twice":
        return v, np.concatenate([f, f, f])
    if name == "far":
        return (v + np.float32(3e4)).astype(np.float32), f
    if name == "large":
        return v * np.float32(1e12), f
    if name == "small":
        return v * np.float32(1e-12), f
    rng = np.random.default_rng(3)      # "noise": no two faces alike, folded over each other
    return (v + rng.normal(0, 0.3, v.shape)).astype(np.float32), f


def _points(v, f, n, seed):
    rng = np.random.default_rng(seed)
    v64 = v.astype(np.float64)
    lo, hi = v64.min(0), v64.max(0)
    size = float((hi - lo).max())
    on = v64[f].mean(1)
    mid = 0.5 * (v64[f[:, 0]] + v64[f[:, 1]])
    near = on[rng.integers(0, len(f), n)] + rng.normal(0, 1e-3 * size, (n, 3))
    wide = lo - size + rng.random((n, 3)) * (hi - lo + 2 * size)
    axis = np.c_[np.zeros((8, 2)), np.linspace(0, 3, 8)] * size + 0.5 * (lo + hi)
    p = np.concatenate([v64[:200], mid[:100], on[:100], axis, near, wide])
    return p[rng.permutation(len(p))].astype(np.float32)


@pytest.mark.parametrize("name", ["faces1", "faces2", "faces3", "faces5", "faces64", "faces65", "fan", "plane", "tube",
                                  "twice", "far", "large", "small", "noise"])
def test_lane_walks_match_oracle(name):
    v, f = _mesh(name)
    gm, om = M.Mesh(v, f), O.Mesh(v, f)
    pr, fwn = M.PointsToMeshProjector(), M.FastWindingNumber(gm)
    pr.updateMeshData(gm)
    pts = _points(v, f, 500, 11)
    size = float((v.max(0) - v.min(0)).max())
    for n in (1, 63, 65, len(pts)):
        for up in (M.FLT_MAX, float(np.float32(0.3 * size) ** 2)):
            say(name, "faces", len(f), "points", n, "limit", up)
            g, o = pr.findProjections(pts[:n], upDistLimitSq=up), om.find_projections(pts[:n], up=up)
            assert np.array_equal(g.view(np.uint8), o.view(np.uint8)), (name, n, up)
    dims, xf, vox = synth.grid_for_mesh(v, (13, 10, 7), expand=1.6)
    for up in (M.FLT_MAX, float(np.float32(0.2 * size) ** 2)):
        g = fwn.calcFromGridWithDistances(dims, xf, M.DistanceToMeshOptions(maxDistSq=up))
        o = om.sdf_grid(dims, xf, O.default_opts(maxDistSq=up))
        assert np.array_equal(np.isnan(g), np.isnan(o)), (name, up)
        ok = ~np.isnan(o)
        assert np.array_equal(np.abs(g[ok]).view(np.uint32), np.abs(o[ok]).view(np.uint32)), (name, up)


def test_lane_walks_match_cooperative_walks():
    """The same calls with a step budget (the wave-cooperative walks) on a mesh of 82 k faces, rigid point
    transform and a limit per query included."""
    import torch
    v, f = synth.bumpy_icosphere(6, 16, 5)
    gm = M.Mesh(v, f)
    pr = M.PointsToMeshProjector()
    pr.updateMeshData(gm)
    n = 40001
    rng = np.random.default_rng(4)
    pts = torch.from_numpy(synth.projection_queries(v, f, n, 6)).cuda()
    lim = torch.from_numpy((rng.random(n) ** 4).astype(np.float32)).cuda()
    xf = np.array([0.96, -0.28, 0, 0.28, 0.96, 0, 0, 0, 1, 0.01, -0.02, 0.03], np.float32)
    out = []
    for budget in (-1, 1, 500):
        gm.set_mode("split_projections", budget)
        for x in (None, xf):
            a = torch.full((n, 8), -5, dtype=torch.int32, device="cuda")
            b = torch.full((n, 8), -5, dtype=torch.int32, device="cuda")
            pr.find_projections_device(pts.data_ptr(), n, a.data_ptr(), ptXf=x)
            pr.find_projections_bounded_device(pts.data_ptr(), n, lim.data_ptr(), b.data_ptr(), ptXf=x)
            torch.cuda.synchronize()
            out.append((a.cpu().numpy(), b.cpu().numpy()))
    for i in (2, 4):
        for k in range(2):
            assert np.array_equal(out[i + k][0], out[k][0]) and np.array_equal(out[i + k][1], out[k][1])


def test_lane_walks_on_more_than_2_23_faces():
    """The stack entries with full refs (trees of more than 2^23 faces) against the per-lane reference form."""
    n = 2060
    rng = np.random.default_rng(1)
    x, y = np.meshgrid(np.arange(n, dtype=np.float32), np.arange(n, dtype=np.float32), indexing="ij")
    v = np.stack([x.ravel(), y.ravel(), rng.random(n * n).astype(np.float32)], 1)
    i, j = (k.ravel() for k in np.meshgrid(np.arange(n - 1), np.arange(n - 1), indexing="ij"))
    a = i * n + j
    f = np.concatenate([np.stack([a, a + n, a + n + 1], 1), np.stack([a, a + n + 1, a + 1], 1)]).astype(np.int32)
    assert len(f) > 1 << 23
    gm = M.Mesh(v, f)
    say("faces", len(f), "depth", gm.depth())
    pr, fwn = M.PointsToMeshProjector(), M.FastWindingNumber(gm)
    pr.updateMeshData(gm)
    pts = (rng.random((3000, 3)) * [n, n, 6] - [0, 0, 3]).astype(np.float32)
    pts[:500] = v[rng.integers(0, len(v), 500)]
    dims, xf, _ = synth.grid_for_mesh(v, (14, 13, 6))
    got = pr.findProjections(pts), fwn.calcFromGridWithDistances(dims, xf, M.DistanceToMeshOptions())
    gm.set_mode("traversal", "per_lane")
    ref = pr.findProjections(pts), fwn.calcFromGridWithDistances(dims, xf, M.DistanceToMeshOptions())
    assert np.array_equal(got[0].view(np.uint8), ref[0].view(np.uint8))
    assert np.array_equal(got[1].view(np.uint32), ref[1].view(np.uint32))
