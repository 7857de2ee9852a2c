"""Up to 2^18 points of a projection are dealt to runs of 256 waves in turn: every point has its record at the edges of runs,
waves and of the range, and a cluster of points that walk long does not end up in a few waves."""
import time

import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import synth

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 255, 256, 257, 2047, 2048, 2049, 4097, 8191, 8193, 65535, 65536, 65537, 131071, 131073, 262143, 262144, 262145]


@pytest.mark.parametrize("n", COUNTS)
def test_every_point_has_its_record(n):
    import torch
    v, f = synth.bumpy_icosphere(3, 5, 2)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    pts = synth.projection_queries(v, f, n, 7)
    xf = np.array([0, 1, 0, -1, 0, 0, 0, 0, 1, 0.1, -0.2, 0.05], np.float32)
    p = torch.from_numpy(pts).cuda()
    limit = torch.rand(n, device="cuda") * 0.2
    out = []
    for form in ("wave_coop", "per_lane"):
        mesh.set_mode("traversal", form)
        r = torch.full((n + 1, 8), -7, dtype=torch.int32, device="cuda")
        proj.find_projections_bounded_device(p.data_ptr(), n, limit.data_ptr(), r.data_ptr(), ptXf=xf)
        torch.cuda.synchronize()
        out.append((proj.findProjections(pts, objXf=xf).view(np.uint8), proj.findProjections(pts, loDistLimitSq=0.01).view(np.uint8),
                    r.cpu().numpy()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert (out[0][2][n] == -7).all()


def test_long_walks_are_spread():
    """A tenth of the time of the form that keeps neighbours together, and a quarter of that of the walks per wave."""
    import torch
    n, faces = 50000, 10000
    a = np.arange(faces) * (2 * np.pi / faces)
    v = np.concatenate([np.stack([np.cos(a), np.sin(a), 0 * a], 1), [[0, 0, 1], [0, 0, -1]]]).astype(np.float32)
    i, j = np.arange(faces), (np.arange(faces) + 1) % faces
    f = np.concatenate([np.stack([i, j, 0 * i + faces], 1), np.stack([j, i, 0 * i + faces + 1], 1)]).astype(np.int32)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    p = torch.from_numpy(np.random.default_rng(1).uniform(-1.2, 1.2, (n, 3)).astype(np.float32)).cuda()
    out = torch.empty((n, 8), dtype=torch.int32, device="cuda")

    def best():
        times = []
        for _ in range(8):
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
    assert lanes < waves
