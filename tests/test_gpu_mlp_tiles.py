"""One training step's kernels at the edges of their 64-row tiles and of the four sums over tiles: the gradient
against the oracle (the bound of the network's other gradient test), Adam's first step from that gradient."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 33, 64, 65, 255, 257, 321, 449])
def test_gradient_and_first_step(n):
    import torch
    import meshlib_amd as M
    rng = np.random.default_rng(n)
    th = np.zeros(MO.NPARAMS, np.float32)
    W = rng.uniform(-0.2, 0.2, size=(MO.LAYERS, MO.HID, MO.HID)).astype(np.float32)
    W[0][:, MO.NFEAT:] = 0
    th[MO.OFF_W:MO.OFF_B] = W.reshape(-1)
    th[MO.OFF_B:MO.OFF_W5] = rng.uniform(-0.1, 0.1, size=MO.LAYERS * MO.HID)
    th[MO.OFF_W5:MO.OFF_B5] = rng.uniform(-0.2, 0.2, size=MO.HID)
    center, scale = np.array([0.2, 0.1, -0.3], np.float32), 1.1
    net = M.DistanceMLP(center, scale, seed=1)
    net.set_params(th)
    pts = rng.uniform(-1.2, 1.2, size=(n, 3)).astype(np.float32)
    lab = rng.uniform(0.0, 0.8, size=n).astype(np.float32)
    dp, dl = torch.from_numpy(pts).cuda(), torch.from_numpy(lab).cuda()
    g = net.gradient(dp, dl).astype(np.float64)
    og = MO.gradient(th, pts, lab, center, scale)
    for sl in (slice(MO.OFF_W, MO.OFF_B), slice(MO.OFF_B, MO.OFF_W5), slice(MO.OFF_W5, MO.OFF_B5),
               slice(MO.OFF_B5, MO.NPARAMS)):
        assert np.linalg.norm(g[sl] - og[sl]) < 2e-2 * max(np.linalg.norm(og[sl]), 1e-12)
    net.train(dp, dl, steps=1, batch=n, lr=1e-2)
    # Adam's first step moves by lr * g / (|g| + eps): where |g| is well above eps = 1e-8, the order of the sum over
    # tiles (about 1e-8 of g) cannot be seen; what is left is the parameters' own rounding
    want = th.astype(np.float64) - 1e-2 * g / (np.abs(g) + 1e-8)
    sure = np.abs(g) > 1e-5
    assert np.max(np.abs(net.get_params() - want)[sure], initial=0.0) < 1e-6
    assert np.all(net.get_params()[g == 0] == th[g == 0])
