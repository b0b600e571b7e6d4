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


@pytest.mark.parametrize("ny,nx", [(1, 64), (3, 128), (17, 192), (67, 64), (128, 1024)])
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
