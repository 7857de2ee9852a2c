"""Points nearest to a vertex of many triangles, all of which are equally far: the record is that of the triangle that the
query's own depth-first walk meets first, whatever their number, and finding it costs no more than testing them."""
import time

import numpy as np
import pytest

import meshlib_amd as M

pytestmark = pytest.mark.gpu


def cone(n, height, turn=None):
    """n triangles around each of two tips above and below a ring"""
    a = np.arange(n) * (2 * np.pi / n)
    v = np.concatenate([np.stack([np.cos(a), np.sin(a), 0 * a], 1), [[0, 0, height], [0, 0, -height]]])
    i, j = np.arange(n), (np.arange(n) + 1) % n
    f = np.concatenate([np.stack([i, j, 0 * i + n], 1), np.stack([j, i, 0 * i + n + 1], 1)])
    if turn is not None:
        q = np.linalg.qr(np.random.default_rng(turn).standard_normal((3, 3)))[0]
        v = v @ q
    return v.astype(np.float32), np.ascontiguousarray(f, np.int32)


def above_tips(v, n, seed):
    """points that are nearest to a tip, and some around the whole cone"""
    rng = np.random.default_rng(seed)
    tips, axis = v[-2:].astype(np.float64), v[-2].astype(np.float64)
    axis = axis / np.linalg.norm(axis)
    k = rng.integers(0, 2, n)
    up = axis * np.where(k == 0, 1, -1)[:, None] * 10.0 ** rng.uniform(-3, 0.5, (n, 1))
    near = tips[k] + up + 0.1 * np.linalg.norm(up, axis=1, keepdims=True) * rng.standard_normal((n, 3))
    return np.concatenate([near, rng.uniform(-1.5, 1.5, (n // 4, 3)) * np.abs(v).max(0)]).astype(np.float32)


@pytest.mark.parametrize("turn", [None, 1, 2])
@pytest.mark.parametrize("n,height", [(3, 1.0), (4, 1.0), (5, 1.0), (9, 10.0), (64, 1.0), (700, 3.0), (4096, 0.5)])
def test_records_match_per_lane(n, height, turn):
    v, f = cone(n, height, turn)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    for count in (40, 1000, 5000):
        pts = above_tips(v, count, n)
        for lo in (0.0, 0.04):
            mesh.set_mode("traversal", "wave_coop")
            got = proj.findProjections(pts, loDistLimitSq=lo)
            mesh.set_mode("traversal", "per_lane")
            want = proj.findProjections(pts, loDistLimitSq=lo)
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), (n, height, turn, count, lo)


def test_ties_cost_no_more_than_their_tests():
    """Against the walks per wave that a step budget selects, which carry the order as keys: 2.5 times their time when every
    tie was put in order as it was met, 1.3 times since, 0.6 with long walks dealt to many waves."""
    import torch
    v, f = cone(3000, 10.0)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    h = np.abs(v).max(0) * 1.2
    n = 50000
    p = torch.from_numpy((h * np.random.default_rng(1).uniform(-1, 1, (n, 3))).astype(np.float32)).cuda()
    out = torch.empty((n, 8), dtype=torch.int32, device="cuda")

    def best():
        times = []
        for _ in range(12):
            torch.cuda.synchronize()
            t = time.perf_counter()
            proj.find_projections_device(p.data_ptr(), n, out.data_ptr())
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t)
        return min(times[2:])

    lanes = best()
    mesh.set_mode("split_projections", 1024)
    waves = best()
    print("lane walks", lanes, "walks per wave", waves, flush=True)
    assert lanes < 1.8 * waves
