"""Steps of single blocks between transmissive and reflective sides, which
read their ghosts where they mirror to: fields with ghosts and every TimeStep
result equal the oracle's bit for bit, at the thinnest blocks, with mixed
sides, and between class-level calls, fixed-dt runs and graph replays."""
import numpy as np
import pytest

import hfo
from hyperflow_amd import case as C
from hyperflow_amd import native

pytestmark = pytest.mark.gpu


def make(nx, ny, scheme, limiter, sides):
    case = C.quad_case(nx, ny, 7, scheme=scheme, limiter=limiter, cfl=0.4)
    for s, k in zip(C.SIDES, sides):
        case.blocks[0].boundaries[s] = {"type": {"T": "Transmissive", "R": "Reflective"}[k]}
    return case, C.perturbed_fields(case, 7)


def same(s, m):
    assert np.array_equal(s.download(0), m.fields(0))
    assert np.array_equal(s.dt_history(), m.dt_log())


@pytest.mark.parametrize("sides", ["TTTT", "RRRR", "RTTR", "TRRT"])
@pytest.mark.parametrize("scheme,limiter,nx,ny", [
    ("Godunov", None, 1, 1), ("Godunov", None, 2, 65), ("Godunov", None, 124, 3), ("MUSCLHancock", "MinBee", 1, 5),
    ("MUSCLHancock", "VanLeer", 2, 2), ("MUSCLHancock", "MinBee", 3, 70), ("MUSCLHancock", "VanLeer", 64, 33),
    ("MUSCLHancock", "MinBee", 121, 62)])
def test_runs_equal_oracle(scheme, limiter, nx, ny, sides):
    case, fields = make(nx, ny, scheme, limiter, sides)
    m = hfo.OracleMesh(case, fields)
    with native.Solver(case) as s:
        s.upload_all(fields)
        for n, graph in ((1, False), (3, False), (2, True), (2, True), (4, False)):
            s.run(n, graph=graph)
            m.run(n)
            same(s, m)
        # the class-level step between device-resident ones
        s.apply_bcs()
        m.apply_bcs()
        dt = s.time_step()
        assert dt == m.time_step()
        s.advance([dt])
        s.run(3)
        with native.Solver(case) as t:   # the same calls step by step
            t.upload_all(fields)
            for _ in range(12):
                t.run(1)
            t.apply_bcs()
            assert t.time_step() == dt
            t.advance([dt])
            for _ in range(3):
                t.run(1)
            assert np.array_equal(s.download(0), t.download(0))
            assert np.array_equal(s.dt_history(), t.dt_history())
            # fixed steps leave the TimeStep counter alone and the next CFL step right
            s.run_fixed(2, 0.1 * dt)
            s.run(2)
            t.run_fixed(2, 0.1 * dt, graph=True)
            t.run(2, graph=True)
            assert np.array_equal(s.download(0), t.download(0))
            assert np.array_equal(s.dt_history(), t.dt_history())
