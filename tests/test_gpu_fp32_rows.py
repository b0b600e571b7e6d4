"""The FP32 row loop, whose window of rows rotates through four names: the
bits do not depend on where items begin and end, and a NaN or an infinity
spreads to the cells that it reaches in FP64."""
import numpy as np
import pytest

from hyperflow_amd import case as C
from hyperflow_amd import native

pytestmark = pytest.mark.gpu


def run(case, fields, steps, precision="fp32", **plan):
    s = native.Solver(case, precision=precision, dt_mode="uniform", **plan)
    s.upload_all(fields)
    s.run(steps)
    out = s.download_all()[0]
    s.close()
    return out


@pytest.mark.parametrize("limiter", ["MinBee", "VanLeer"])
@pytest.mark.parametrize("ny", [1, 2, 3, 4, 5, 6, 9, 63])
def test_items_of_any_length_give_the_same_bits(limiter, ny):
    case = C.quad_case(131, ny, 5, scheme="MUSCLHancock", limiter=limiter, cfl=0.4, bc="Reflective")
    fields = C.perturbed_fields(case, 3)
    ref = run(case, fields, 5, tile_rows=64, tail_rows=64)
    assert np.isfinite(ref).all()
    for rows in (1, 2, 3, 4, 5, 7):
        assert np.array_equal(run(case, fields, 5, tile_rows=rows, tail_rows=rows), ref)


@pytest.mark.parametrize("limiter", ["MinBee", "VanLeer"])
@pytest.mark.parametrize("var", range(4))
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf], ids=["nan", "inf", "-inf"])
def test_values_that_are_not_finite_spread_as_in_fp64(limiter, var, value):
    case = C.quad_case(90, 40, 5, scheme="MUSCLHancock", limiter=limiter, cfl=0.4, bc="Transmissive")
    fields = C.perturbed_fields(case, 3)
    fields[0][var, 20, 30] = value
    with np.errstate(all="ignore"):
        a, b = run(case, fields, 1), run(case, fields, 1, precision="fp64")
    assert np.array_equal(np.isfinite(a), np.isfinite(b))
