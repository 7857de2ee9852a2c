"""The batch's work units at the edges of their dealing: one unit, fewer units than XCDs or than a run, many items of one
unit each, a run that ends inside an item; with and without a range of units per XCD."""
import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import synth

pytestmark = pytest.mark.gpu


# (items, points per item) with a 5x4x6 grid (4 units) on every third item
@pytest.mark.parametrize("count,points", [(1, 1), (1, 64 * 64), (1, 64 * 64 * 8 + 1), (5, 65), (71, 1), (130, 63), (9, 64 * 60)])
@pytest.mark.parametrize("split", [0, 1])
def test_every_unit_runs_once(count, points, split):
    import torch
    v, f = synth.bumpy_icosphere(2, 3, 4)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    fwn = M.FastWindingNumber(mesh)
    dims, xf, _ = synth.grid_for_mesh(v, (5, 4, 6))
    sdf = torch.from_numpy(np.asarray(fwn.calcFromGridWithDistances(dims, xf, M.DistanceToMeshOptions()))).cuda()
    pts = torch.from_numpy(synth.projection_queries(v, f, count * points, 8)).cuda()
    rec = torch.full((count * points, 8), -7, dtype=torch.int32, device="cuda")
    proj.find_projections_device(pts.data_ptr(), count * points, rec.data_ptr())
    got = torch.full_like(rec, -7)
    vol = torch.full((count, sdf.numel()), -7.0, device="cuda")
    torch.cuda.synchronize()
    items = []
    for i in range(count):
        it = {"mesh": mesh, "d_pts": pts[i * points:].data_ptr(), "n": points, "d_proj": got[i * points:].data_ptr()}
        if i % 3 == 0:
            it.update(dims=dims, xf=xf, d_sdf=vol[i].data_ptr())
        items.append(it)
    batch = M.Batch()
    batch.set_config(4, split)
    batch.run(items)
    torch.cuda.synchronize()
    assert torch.equal(got, rec)
    for i in range(count):
        assert torch.equal(vol[i], sdf.reshape(-1)) if i % 3 == 0 else bool((vol[i] == -7).all())
