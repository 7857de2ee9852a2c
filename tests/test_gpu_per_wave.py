"""Launches that spread their queries over partly filled waves: a query's result does not depend on how many
others share its wave, so every small call gives the bits that the same queries have in a call of full waves."""
import functools

import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import synth

pytestmark = pytest.mark.gpu

FULL = (1 << 19) + 64 * 5 + 3          # full waves in every form, with a ragged last one


@functools.lru_cache(None)
def full_call():
    import torch
    v, f = synth.bumpy_icosphere(4, 8, 5)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    fwn = M.FastWindingNumber(mesh)
    pts = torch.from_numpy(synth.projection_queries(v, f, FULL, 3)).cuda()
    pts = pts[torch.randperm(FULL, device="cuda", generator=torch.Generator("cuda").manual_seed(1))].contiguous()
    rec = torch.empty((FULL, 8), dtype=torch.int32, device="cuda")
    wn = torch.empty(FULL, dtype=torch.int32, device="cuda")
    proj.find_projections_device(pts.data_ptr(), FULL, rec.data_ptr())
    fwn.fwn_vector_device(pts.data_ptr(), FULL, 2.0, wn.data_ptr())
    torch.cuda.synchronize()
    return mesh, proj, fwn, pts, rec, wn


# the ends of the ranges of 1, 2, 4 .. 64 queries a wave, and odd remainders
@pytest.mark.parametrize("n", [1, 63, 2048, 2049, 4096, 4097, 8193, 16385, 32769, 65537, 131073, 262144, 262145, 1 << 19])
def test_points_in_partly_filled_waves(n):
    import torch
    _, proj, fwn, pts, rec, wn = full_call()
    r = torch.full((n, 8), -7, dtype=torch.int32, device="cuda")
    w = torch.full((n,), -7, dtype=torch.int32, device="cuda")
    proj.find_projections_device(pts.data_ptr(), n, r.data_ptr())
    fwn.fwn_vector_device(pts.data_ptr(), n, 2.0, w.data_ptr())
    assert torch.equal(r, rec[:n])
    assert torch.equal(w, wn[:n])


# slabs of one grid of full waves; the depth of the slab sets the voxels a wave takes
@pytest.mark.parametrize("layers", [1, 4, 9, 33])
def test_grid_slabs_in_partly_filled_waves(layers):
    import torch
    mesh, _, fwn, _, _, _ = full_call()
    v, _ = synth.bumpy_icosphere(4, 8, 5)
    dims, xf, _ = synth.grid_for_mesh(v, (71, 66, 80))
    opts = M.DistanceToMeshOptions()
    nx, ny, nz = (int(d) for d in dims)
    for call in (lambda out, a, b: fwn.sdf_grid_device(dims, xf, opts, out.data_ptr(), zBegin=a, zEnd=b),
                 lambda out, a, b: fwn.fwn_grid_device(dims, xf, 2.0, out.data_ptr(), zBegin=a, zEnd=b)):
        whole = torch.full((nz, ny, nx), -7, dtype=torch.int32, device="cuda")
        call(whole, 0, nz)
        for a in (0, 37):
            part = torch.full((layers, ny, nx), -7, dtype=torch.int32, device="cuda")
            call(part, a, a + layers)
            assert torch.equal(part, whole[a:a + layers])


@pytest.mark.parametrize("level", [0, 1, 3])
def test_self_intersections_in_partly_filled_waves(level):
    v, f = synth.bumpy_icosphere(level, 8, 5)
    v2 = np.concatenate([v, v * np.float32(0.5) + np.float32(0.7)])      # two shells that cross
    f2 = np.concatenate([f, f + len(v)]).astype(np.int32)
    mesh = M.Mesh(v2, f2)
    fwn = M.FastWindingNumber(mesh)
    got = np.asarray(fwn.calcSelfIntersections(2.0))
    M.set_traversal("per_lane")
    try:
        one = np.asarray(fwn.calcSelfIntersections(2.0))
    finally:
        M.set_traversal("wave_coop")
    assert np.array_equal(got, one)


def test_winding_numbers_on_more_than_2_23_faces():
    """Places of records beyond 32-bit byte offsets: winding numbers of points against the per-lane form."""
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
        # the wave form's square roots and quotients may be off by one unit in about one of 10^7 cases
        assert np.allclose(g, w, rtol=0, atol=1e-5)
