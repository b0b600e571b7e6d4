"""Plans of the guess and check launches over blocks whose wave-speed maxima
lie in one to eight slots, in problems of more than 64 blocks and in several
problems of one context: bit for bit the CPU oracle's fields and TimeStep
results, also where the check launch computes."""
import numpy as np
import pytest

import context_probe
import gpu_util as G
from hyperflow_amd import case as C

pytestmark = pytest.mark.gpu


def row_of_blocks(count, nx, ny, limiter):
    """count blocks side by side, listed from the right to the left."""
    base = C.quad_case(8, 8, 3, scheme="MUSCLHancock", limiter=limiter, cfl=0.5)
    wall, inner = {"type": "Reflective"}, lambda b: {"type": "Internal", "block": b}
    base.blocks = [C.Block((count - 1 - k) / count, (count - k) / count, 0.0, 1.0, nx, ny,
                           {"bottom": wall, "top": wall, "right": inner(k - 1) if k else wall,
                            "left": inner(k + 1) if k + 1 < count else wall}) for k in range(count)]
    return base


def check(cases, ways, steps, computed=None):
    """computed: tallies of fixup_stats() that must have counted blocks."""
    data = [(c, C.perturbed_fields(C.Case(**{**c.__dict__, "initial_condition": C.quad_case(8, 8, 2).initial_condition}), 2))
            for c in cases]
    ref = [G.oracle_run(c, f, steps) for c, f in data]
    s, out, hist = G.gpu_run(cases, [U for _, f in data for U in f], steps)
    got, fixups = context_probe.ways(s), s.fixup_stats()
    s.close()
    assert ways is None or got == ways
    assert all(fixups[k] > 0 for k in computed or ()), fixups
    assert np.array_equal(hist, ref[0][1])
    for a, b in zip(out, [U for r in ref for U in r[0]]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,ways", [(10, 1), (17, 2), (40, 4), (97, 8)])
@pytest.mark.parametrize("limiter", ["MinBee", "VanLeer"])
def test_channel(n, ways, limiter):
    check([C.step_channel(n, limiter, 0.5)], ways, 16)


def test_more_than_64_blocks():
    check([row_of_blocks(70, 20, 170, "VanLeer")], 2, 13)


def test_several_problems():
    check([C.step_channel(97, "MinBee", 0.5), row_of_blocks(3, 33, 20, "MinBee"), C.step_channel(17, "MinBee", 0.5)], 8, 13)


@pytest.mark.parametrize("sizes", [(20, 170, 70), (33, 20, 9), (61, 97, 5), (128, 64, 12)])
@pytest.mark.parametrize("count", [1, 3])
def test_check_launch_that_computes(sizes, count):
    """Rows of blocks in which the check launch recomputes blocks, round after
    round, with fewer waves than are resident (one per item of a round)."""
    nx, ny, blocks = sizes
    cases = [row_of_blocks(blocks, nx, ny, "VanLeer")] + [row_of_blocks(3 + k, 33, 20, "VanLeer") for k in range(count - 1)]
    check(cases, None, 40, ("check",))
