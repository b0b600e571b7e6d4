"""Work plans of one round of short items and their spread wave-speed maxima:
sizes around strips, edge bands cut into several items and slots per block,
bit for bit the CPU oracle's fields and TimeStep results."""
import numpy as np
import pytest

import gpu_util as G
from hyperflow_amd import case as C

pytestmark = pytest.mark.gpu


def check(case, fields, steps):
    ref, calls, _ = G.oracle_run(case, fields, steps)
    s, out, hist = G.gpu_run(case, fields, steps)
    s.close()
    assert np.array_equal(hist, calls)
    for a, b in zip(out, ref):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("scheme,limiter,nx,ny", [
    ("Godunov", None, 1, 130), ("Godunov", None, 62, 1), ("Godunov", None, 63, 700), ("Godunov", None, 400, 37),
    ("MUSCLHancock", "MinBee", 2, 3), ("MUSCLHancock", "MinBee", 61, 300), ("MUSCLHancock", "VanLeer", 90, 200),
    ("MUSCLHancock", "VanLeer", 91, 61), ("MUSCLHancock", "MinBee", 300, 5), ("MUSCLHancock", "VanLeer", 330, 410)])
def test_single_block(scheme, limiter, nx, ny):
    case = C.quad_case(nx, ny, 5, scheme=scheme, limiter=limiter, cfl=0.4)
    check(case, C.perturbed_fields(case, 5), 12)


@pytest.mark.parametrize("n", [17, 65, 97])
def test_channel(n):
    case = C.step_channel(n, "VanLeer", 0.5)
    check(case, C.perturbed_fields(C.Case(**{**case.__dict__, "initial_condition": C.quad_case(
        4, 4, 2).initial_condition}), 2), 14)
