"""The network's gradients and forward pass at the sizes where its launches
are cut differently: one row, ragged rows, several strips, and images large
enough for more rows per workgroup, against the CPU reference."""
import numpy as np
import pytest

import cnn_ref as R
from hyperflow_amd import native
from test_gpu_learned import NORM, OFFS, dev, state

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("ny,nx", [(1, 64), (3, 128), (17, 192), (67, 64), (251, 256), (128, 1024)])
def test_gradients_at_sizes(ny, nx):
    net = native.Net(**NORM, seed=ny)
    p = net.get_params()
    u = state(ny, ny, nx).astype(np.float32)
    t = (u + np.random.default_rng(nx).normal(scale=0.01, size=u.shape)).astype(np.float32)
    L, g = net.gradients(dev(u), dev(t))
    Lr, gr = R.gradients(p, u, t, emulate=True, **NORM)
    assert abs(L - Lr) <= 1e-4 * Lr
    for l in range(5):
        a = slice(OFFS[l], OFFS[l + 1])
        assert np.linalg.norm(g[a] - gr[a]) < 1e-2 * np.linalg.norm(gr[a])


@pytest.mark.parametrize("ny,nx", [(1, 64), (4, 64), (5, 128), (66, 192), (300, 64), (9, 704)])
def test_forward_at_sizes(ny, nx):
    """Strips of 80 columns and their chunks of rows: images narrower than a
    strip, ending inside one, of one row and of several chunks; every pixel,
    the edges above all, within the bounds of the full-size test."""
    net = native.Net(**NORM, seed=nx)
    u = state(ny + nx, ny, nx).astype(np.float32)
    y = torch.full((4, ny, nx), float("nan"), device="cuda")
    net.forward(dev(u), y)
    net.synchronize()
    torch.cuda.synchronize()
    yr, _ = R.forward(net.get_params(), u, NORM["in_mean"], NORM["in_scale"], emulate=True)
    yg = y.cpu().numpy().astype(np.float64)
    assert np.max(np.abs(yg - yr)) < 2e-3 * np.max(np.abs(yr))
    assert np.mean(np.abs(yg - yr)) < 2e-4 * np.mean(np.abs(yr))
