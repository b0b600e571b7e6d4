"""FP64 rows at the ends of the range in which the sweeps take the shortened
divisions (q64 in hf_physics.h): bit for bit the CPU oracle's results, signed
zeros included, whether an item stays in range, leaves it on its first row or
somewhere in its middle."""
import numpy as np
import pytest

import gpu_util as G
from hyperflow_amd import case as C

pytestmark = pytest.mark.gpu


def fields_of(case, what):
    """perturbed_fields with a band of rows and a band of columns changed."""
    fields = C.perturbed_fields(case, 3)
    g = case.ghost
    for b, U in zip(case.blocks, fields):
        rows, cols = slice(g + b.ny // 3, g + b.ny // 3 + 7), slice(g + b.nx // 2, g + b.nx // 2 + 5)
        for band in ((slice(None), rows, slice(g, g + b.nx)), (slice(None), slice(g, g + b.ny), cols)):
            V = U[band]
            kind, e = what
            if kind == "state":            # the whole state scaled: rho and E leave their ranges
                V *= 2.0 ** e
            elif kind == "momentum":       # tiny momenta, down to subnormals
                V[1:3] *= 2.0 ** e
            elif kind == "one":            # one tiny momentum beside an exact zero
                V[1] = 0.0
                V[2] *= 2.0 ** e
            elif kind == "zero":           # zeros of both signs
                V[1], V[2] = 0.0, -0.0
            elif kind == "energy":
                V[3] *= 2.0 ** e
    return fields


WHAT = [("state", -58), ("state", -62), ("state", 38), ("state", 42), ("momentum", -400), ("momentum", -797),
        ("momentum", -803), ("momentum", -1060), ("one", -500), ("one", -900), ("zero", 0), ("energy", -4),
        ("energy", -98)]


@pytest.mark.parametrize("what", WHAT, ids=[f"{k}{e}" for k, e in WHAT])
@pytest.mark.parametrize("scheme,limiter,bc", [("Godunov", None, "Reflective"), ("MUSCLHancock", "MinBee", "Transmissive"),
                                               ("MUSCLHancock", "VanLeer", "Reflective")])
def test_bits_equal_oracle(scheme, limiter, bc, what):
    case = C.quad_case(83, 61, 3, scheme=scheme, limiter=limiter, cfl=0.4, bc=bc)   # 60 + 23: a transposed band too
    fields = fields_of(case, what)
    with np.errstate(all="ignore"):
        ref, calls, _ = G.oracle_run(case, fields, 6)
    s, out, hist = G.gpu_run(case, fields, 6)
    s.close()
    assert np.array_equal(hist, calls)
    a, b = out[0], ref[0]
    nan = np.isnan(b)
    assert np.array_equal(np.isnan(a), nan)
    assert np.array_equal(np.where(nan, 0, a).view(np.int64), np.where(nan, 0, b).view(np.int64))
