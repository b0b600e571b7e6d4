"""Large downloads, which the device packs into pinned pieces that several
threads carry to the caller's array: every value where the caller put it, at
sizes around the threshold and the pieces' ends, in both arithmetics, several
blocks and several threads at once."""
import threading

import numpy as np
import pytest

from hyperflow_amd import case as C
from hyperflow_amd import native

pytestmark = pytest.mark.gpu

# [4][ny+4][nx+4] values: just below and at 2^20 (one pageable copy), then pieces
# of 2^18 with short and nearly whole last ones, and rows longer than a piece
SIZES = [(508, 507), (508, 508), (509, 509), (507, 1020), (1500, 177), (300001, 1)]


def numbered(case):
    out = []
    for i, b in enumerate(case.blocks):
        shape = (4, b.ny + 2 * case.ghost, b.nx + 2 * case.ghost)
        n = int(np.prod(shape))
        out.append((1.0 + i + np.arange(n) / n).astype(np.float32).astype(np.float64).reshape(shape))
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("size", SIZES, ids=[f"{x}x{y}" for x, y in SIZES])
def test_values_come_back_in_place(size, precision):
    case = C.quad_case(*size, 3, scheme="MUSCLHancock", limiter="VanLeer", cfl=0.4, bc="Transmissive")
    s = native.Solver(case, precision=precision)
    fields = numbered(case)
    s.upload_all(fields)
    for _ in range(2):
        for a, b in zip(s.download_all(), fields):
            assert np.array_equal(a, b)
    s.close()


def test_threads_download_their_own_contexts():
    case = C.quad_case(700, 600, 3, scheme="MUSCLHancock", limiter="VanLeer", cfl=0.4, bc="Transmissive")
    solvers = [native.Solver(case, precision="fp64") for _ in range(3)]
    fields = numbered(case)[0]
    bad = []

    def work(i):
        mine = fields + i
        for _ in range(3):
            solvers[i].upload(0, mine)
            if not np.array_equal(solvers[i].download(0), mine):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for s in solvers:
        s.close()
