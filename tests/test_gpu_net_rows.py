"""The network's streaming forward pass with many rows per workgroup: every
pixel's bits are those of short images of the same rows (four rows per
workgroup, the ones compared with the CPU reference elsewhere; 14 at the widest),
as a pixel's operations do not depend on where its workgroup began.  The
correction in place likewise; gradients against the CPU reference."""
import numpy as np
import pytest

import cnn_ref as R
from hyperflow_amd import case as C
from hyperflow_amd import native
from test_gpu_learned import NORM, OFFS, dev, state

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

HALO = 5   # rows that a pixel of the output reaches


def rows_per_workgroup(nx, ny):
    """launch_net's rule."""
    strips = -(-nx // 80)
    return min(128, max(4, -(-ny // (256 // strips if strips < 256 else 1))))


def forward(net, u):
    y = torch.full(u.shape, float("nan"), device="cuda")
    net.forward(u, y)
    net.synchronize()
    return y


# (rows, columns, rows per workgroup): ragged last chunks, and the most rows
# per workgroup (129 strips: one chunk for each, of 128 rows, then one of 3)
SIZES = [(200, 1536, 17), (333, 1024, 18), (1100, 64, 5), (131, 10304, 128)]


@pytest.mark.parametrize("ny,nx,rows", SIZES)
def test_forward_in_long_chunks_equals_short_ones(ny, nx, rows):
    assert rows_per_workgroup(nx, ny) == rows
    net = native.Net(**NORM, seed=nx)
    u = dev(state(ny + nx, ny, nx))
    y = forward(net, u)
    assert bool(torch.isfinite(y).all())
    h = 14 if nx > 10000 else 40   # rows of a short image
    assert rows_per_workgroup(nx, h) == (14 if nx > 10000 else 4)
    step = h - 2 * HALO
    for y0 in range(0, ny, step):
        lo, hi = max(0, y0 - HALO), min(ny, y0 + step + HALO)
        part = forward(net, u[:, lo:hi].contiguous())
        y1 = min(ny, y0 + step)
        assert torch.equal(part[:, y0 - lo:y1 - lo], y[:, y0:y1]), (y0, y1)


@pytest.mark.parametrize("ny,nx,rows", SIZES[:3])
@pytest.mark.parametrize("max_output", [0.0, 0.5])
def test_correction_in_long_chunks(ny, nx, rows, max_output):
    case = C.quad_case(nx, ny, 6, scheme="MUSCLHancock", limiter="VanLeer", cfl=0.5)
    g = case.ghost
    net = native.Net(in_mean=[1, 0, 0, 2.5], in_scale=[1, 1, 1, 1], out_scale=[0.5, 0.1, 0.1, 1.0], gamma=1.4,
                     shock_threshold=0.2, seed=12, max_output=max_output)
    p = net.get_params()
    p[OFFS[4] + 9 * 32 * 4 + 0] = -0.3      # push the density down so some cells go non-positive
    net.set_params(p)
    with native.Solver(case, precision="fp32", dt_mode="uniform") as s:
        s.upload(0, C.perturbed_fields(case, 6)[0])
        s.run(2)
        U = s.download(0)[:, g:-g, g:-g].astype(np.float32)
        y = forward(net, dev(U)).cpu().numpy()
        nfb = s.correct(net, count=True)
        out = s.download(0)[:, g:-g, g:-g].astype(np.float32)
    exp, bad = R.apply_correction(U, y, net.desc["out_scale"], 1.4, 0.2, dtype=np.float32, max_output=max_output)
    assert 0 < nfb < U[0].size and nfb == int(bad.sum())
    np.testing.assert_array_equal(out, exp.astype(np.float32))


def test_gradients_with_stored_activations():
    ny, nx = 100, 1536
    assert rows_per_workgroup(nx, ny) == 9
    net = native.Net(**NORM, seed=4)
    u = state(4, ny, nx).astype(np.float32)
    t = (u + np.random.default_rng(nx).normal(scale=0.01, size=u.shape)).astype(np.float32)
    L, g = net.gradients(dev(u), dev(t))
    Lr, gr = R.gradients(net.get_params(), u, t, emulate=True, **NORM)
    assert abs(L - Lr) <= 1e-4 * Lr
    for l in range(5):
        a = slice(OFFS[l], OFFS[l + 1])
        assert np.linalg.norm(g[a] - gr[a]) < 1e-2 * np.linalg.norm(gr[a])
