"""Queries far from the mesh: the limit's relative slack would hold most of it, so beyond a distance that depends on the
mesh lanes walk over boxes.  Records are the oracle's bit for bit on both sides of that line, also in waves that hold near and
far queries, with limits and with low limits, and a query visits a small part of the tree at every distance."""
import numpy as np
import pytest

import meshlib_amd as M
from meshlib_amd import synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def directions(n, seed):
    d = np.random.default_rng(seed).standard_normal((n, 3))
    return d / np.linalg.norm(d, axis=1, keepdims=True)


@pytest.mark.parametrize("faces", [1, 2, 300, 1280])
def test_far_queries_match_oracle(faces):
    v, f = synth.bumpy_icosphere(3, 5, 2)
    f = np.ascontiguousarray(f[:faces])
    gm, om = M.Mesh(v, f), O.Mesh(v, f)
    proj, fwn = M.PointsToMeshProjector(), M.FastWindingNumber(gm)
    proj.updateMeshData(gm)
    rng = np.random.default_rng(5)
    pts = np.concatenate([directions(150, k) * 10.0 ** k for k in range(0, 13, 2)] + [synth.projection_queries(v, f, 300, 3)])
    pts = pts[rng.permutation(len(pts))].astype(np.float32)
    for up in (M.FLT_MAX, 1e10):
        for lo in (0.0, 0.5, 1e9):
            g = proj.findProjections(pts, upDistLimitSq=up, loDistLimitSq=lo)
            o = om.find_projections(pts, up=up, lo=lo)
            assert np.array_equal(g.view(np.uint8), o.view(np.uint8)), (faces, up, lo)
    # a grid with one corner at the mesh and steps of 1e4 and 1e7
    for step in (1e4, 1e7):
        dims, xf = np.array([9, 7, 6], np.int32), np.array([step, 0, 0, 0, step, 0, 0, 0, step, 0.1, 0.2, 0.3], np.float32)
        g = fwn.calcFromGridWithDistances(dims, xf, M.DistanceToMeshOptions())
        o = om.sdf_grid(dims, xf)
        assert np.array_equal(np.abs(g).view(np.uint32), np.abs(o).view(np.uint32)), (faces, step)


@pytest.mark.parametrize("distance,visits", [(1e3, 1200), (1e5, 3600), (1e6, 1000), (1e12, 1000)])
def test_far_queries_visit_a_small_part(distance, visits):
    """20,479 nodes; with twice the slack 4,800 at 1e5 and, without the walk over boxes, all from 1e6 on."""
    import torch
    v, f = synth.bumpy_icosphere(5, 8, 1)
    mesh = M.Mesh(v, f)
    proj = M.PointsToMeshProjector()
    proj.updateMeshData(mesh)
    counts = torch.zeros(M.STAT_LAUNCHES * M.STAT_STRIDE, dtype=torch.int64, device="cuda")
    mesh.set_stats(counts.data_ptr())
    pts = torch.from_numpy((directions(1000, 1) * distance).astype(np.float32)).cuda()
    out = torch.empty((1000, 8), dtype=torch.int32, device="cuda")
    proj.find_projections_device(pts.data_ptr(), 1000, out.data_ptr())
    torch.cuda.synchronize()
    each = counts[M.STAT_NAMES.index("lane_visits")].item() / 1000
    print("distance", distance, "visits", each, flush=True)
    assert 0 < each < visits
