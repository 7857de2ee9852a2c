"""Margins of the lane walks' bounds: flat oblique patches, small against their coordinates, which lie just above a power of
two, so that the roundings of a node's centre and of the leaf test's closest point add up.  Every query's limit is the next
float above its distance, so a bound that is too large by the least amount loses the only leaf that can answer."""
import numpy as np
import pytest

import meshlib_amd as M

pytestmark = pytest.mark.gpu


def patches(n, base, seed):
    """n flat quads with normals near (1, 1, 1) / sqrt(3), corners at base .. 1.05 base"""
    rng = np.random.default_rng(seed)
    nrm = 1 + 0.1 * rng.uniform(-1, 1, (n, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    e = np.cross(nrm, rng.standard_normal((n, 3)))
    e /= np.linalg.norm(e, axis=1, keepdims=True)
    f = np.cross(nrm, e)
    size = base * 10.0 ** rng.uniform(-4.5, -2.5, (n, 1))
    c = base * (1 + 0.05 * rng.random((n, 3)))
    v = np.stack([c - size * e, c - size * f, c + size * e, c + size * f], 1).reshape(-1, 3)
    i = 4 * np.arange(n)
    tri = np.concatenate([np.stack([i, i + 1, i + 2], 1), np.stack([i, i + 2, i + 3], 1)])
    k = rng.integers(0, n, 40 * n)
    at = c[k] + size[k] * (rng.uniform(-0.5, 0.5, (len(k), 1)) * e[k] + rng.uniform(-0.5, 0.5, (len(k), 1)) * f[k])
    pts = at + size[k] * 10.0 ** rng.uniform(-4, 0, (len(k), 1)) * rng.choice([-1, 1], (len(k), 1)) * nrm[k]
    return v.astype(np.float32), np.ascontiguousarray(tri, np.int32), pts.astype(np.float32)


@pytest.mark.parametrize("base", [1.0, 32.0])
def test_limits_just_above_the_distance(base):
    import torch
    v, f, pts = patches(20000, base, 7)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    n = len(pts)
    p = torch.from_numpy(pts).cuda()

    def records(limit=None):
        r = torch.full((n, 8), -5, dtype=torch.int32, device="cuda")
        if limit is None:
            proj.find_projections_device(p.data_ptr(), n, r.data_ptr())
        else:
            proj.find_projections_bounded_device(p.data_ptr(), n, limit.data_ptr(), r.data_ptr())
        torch.cuda.synchronize()
        return r

    mesh.set_mode("traversal", "per_lane")
    want = records()
    mesh.set_mode("traversal", "wave_coop")
    limit = torch.nextafter(want[:, 7].contiguous().view(torch.float32), torch.tensor(float("inf"), device="cuda"))
    got, bounded = records(), records(limit)
    wrong = (got != want).any(1).sum().item(), (bounded != want).any(1).sum().item()
    print("coordinates", base, "queries", n, "wrong", wrong, flush=True)
    assert wrong == (0, 0)
