"""FP64 rows at the ends of the range in which the sweeps take the shortened
divisions (q64 in hf_physics.h): bit for bit the CPU oracle's results, signed
zeros included, whether an item stays in range, leaves it on its first row or
somewhere in its middle."""
import numpy as np
import pytest

import gpu_util as G
import hfo
from hyperflow_amd import case as C
from hyperflow_amd import uns

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


def bits_equal(a, b):
    nan = np.isnan(b)
    return np.array_equal(np.isnan(a), nan) and np.array_equal(np.where(nan, 0, a).view(np.int64),
                                                               np.where(nan, 0, b).view(np.int64))


@pytest.mark.parametrize("what", WHAT + [("rest", 0), ("vacuum", 0)], ids=[f"{k}{e}" for k, e in WHAT] + ["rest", "vacuum"])
def test_unstructured_bits_equal_oracle(what):
    """Cells of an unstructured mesh, some of them out of range beside cells
    in range: the wave's results are the oracle's either way."""
    kind, e = what
    quads, codes = uns.box(23, 17, code=uns.TRANSMISSIVE, skew=0.35)
    codes[::5, 1] = np.where(codes[::5, 1] != 0, uns.REFLECTIVE, 0)
    codes[:23, 0] = uns.INLET
    rng = np.random.default_rng(7)
    W = np.stack([rng.uniform(0.3, 2.0, len(quads)), rng.uniform(-1, 1, len(quads)), rng.uniform(-1, 1, len(quads)),
                  rng.uniform(0.2, 3.0, len(quads))], axis=1)
    inlet = uns.prim_to_cons([1.5, 0.8, 0.1, 1.2], 1.4)
    if kind == "rest":          # one state at rest everywhere: speeds of exactly zero
        W[:] = [1.2, 0.0, 0.0, 0.7]
        inlet = uns.prim_to_cons([1.2, 0.0, 0.0, 0.7], 1.4)
    V = np.array([uns.prim_to_cons(w, 1.4) for w in W])
    band = V[150:157]           # crosses the middle of a wave's cells
    if kind == "state":
        band *= 2.0 ** e
    elif kind == "momentum":
        band[:, 1:3] *= 2.0 ** e
    elif kind == "one":
        band[:, 1] = 0.0
        band[:, 2] *= 2.0 ** e
    elif kind == "zero":
        band[:, 1], band[:, 2] = 0.0, -0.0
    elif kind == "energy":
        band[:, 3] *= 2.0 ** e
    elif kind == "vacuum":      # no density: quotients by zero
        band[:] = 0.0
    s = uns.UnsSolver(quads, codes, inlet, 1.4, 0.4)
    o = hfo.UnsOracle(quads, codes, inlet, 1.4, 0.4)
    s.upload(V)
    o.set_fields(V)
    s.run(6)
    with np.errstate(all="ignore"):
        dts = o.run(6)
    assert bits_equal(np.array(s.dt_history()), np.array(dts))
    assert bits_equal(s.download(), o.fields())
    s.close()
