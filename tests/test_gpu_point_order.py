"""The spatial ordering of query points: whatever the number and place of the points, every one of them is answered
once, with the answer it has on its own."""
import functools

import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import synth

pytestmark = pytest.mark.gpu

BASE = 97


@functools.lru_cache(None)
def base():
    """97 points (inside, outside, far outside the mesh's box, on its corners) and their answers one by one"""
    import torch
    v, f = synth.bumpy_icosphere(3, 4, 9)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    fwn = M.FastWindingNumber(mesh)
    pts = synth.projection_queries(v, f, BASE, 2)
    pts[0], pts[1], pts[2] = v.min(0), v.max(0), (1e6, -3e5, 7.0)
    pts = torch.from_numpy(pts).cuda()
    rec = torch.empty((BASE, 8), dtype=torch.int32, device="cuda")
    wn = torch.empty(BASE, dtype=torch.int32, device="cuda")
    for i in range(BASE):
        proj.find_projections_device(pts[i].data_ptr(), 1, rec[i].data_ptr())
        fwn.fwn_vector_device(pts[i].data_ptr(), 1, 2.0, wn[i:].data_ptr())
    torch.cuda.synchronize()
    return proj, fwn, pts, rec, wn


# the ends of each range of cells, of the points per thread and of the counting sort
@pytest.mark.parametrize("n", [1, 511, 512, 2049, 8192, 8193, 32768, 32769, 262144, 262145, (1 << 21) - 7, 1 << 21, (1 << 21) + 1])
@pytest.mark.parametrize("cloud", ["spread", "one", "two"])
def test_every_point_is_answered(n, cloud):
    import torch
    proj, fwn, pts, rec, wn = base()
    kinds = {"spread": BASE, "one": 1, "two": 2}[cloud]
    idx = torch.from_numpy(np.random.Generator(np.random.PCG64(n)).integers(0, kinds, n)).cuda()
    if cloud == "one":
        idx += 5
    q = pts[idx].contiguous()
    r = torch.full((n, 8), -7, dtype=torch.int32, device="cuda")
    w = torch.full((n,), -7, dtype=torch.int32, device="cuda")
    proj.find_projections_device(q.data_ptr(), n, r.data_ptr())
    fwn.fwn_vector_device(q.data_ptr(), n, 2.0, w.data_ptr())
    assert torch.equal(r, rec[idx])
    assert torch.equal(w, wn[idx])
