"""Captured step loops: one graph serves every run of its length (two where
the length is odd, by the buffer that the run starts from), and replays mixed
with other runs give the oracle's bits."""
import numpy as np
import pytest

import context_probe
import hfo
from hyperflow_amd import case as C
from hyperflow_amd import native

pytestmark = pytest.mark.gpu


def make(kind):
    if kind == "channel":
        case = C.step_channel(20, "MinBee", 0.5)
        like = C.Case(**{**case.__dict__, "initial_condition": C.quad_case(4, 4, 2).initial_condition})
        return case, C.perturbed_fields(like, 2)
    scheme, limiter = ("Godunov", None) if kind == "godunov" else ("MUSCLHancock", "VanLeer")
    case = C.quad_case(150, 90, 7, scheme=scheme, limiter=limiter, cfl=0.4)
    return case, C.perturbed_fields(case, 7)


@pytest.mark.parametrize("kind", ["godunov", "muscl", "channel"])
@pytest.mark.parametrize("n,held", [(20, 1), (7, 2), (6, 1), (1, 2)])
def test_a_length_is_captured_once(kind, n, held):
    case, fields = make(kind)
    m = hfo.OracleMesh(case, fields)
    with native.Solver(case) as s:
        s.upload_all(fields)
        for _ in range(10):
            s.run(n, graph=True)
        m.run(10 * n)
        assert context_probe.graphs(s) == held
        # eager runs and another length between replays
        for k, graph in ((2, False), (n, True), (5, False), (n, True), (4, True), (n, True)):
            s.run(k, graph=graph)
            m.run(k)
            assert all(np.array_equal(s.download(b), m.fields(b)) for b in range(len(fields)))
        assert np.array_equal(s.dt_history(), m.dt_log())


def test_fixed_steps_are_captured_once():
    case, fields = make("muscl")
    dt = 2e-4
    with native.Solver(case) as s, native.Solver(case) as t:
        for x in (s, t):
            x.upload_all(fields)
        for _ in range(6):
            s.run_fixed(5, dt, graph=True)
            s.run(4, graph=True)
            t.run_fixed(5, dt)
            t.run(4)
        assert context_probe.graphs(s) == 4
        assert np.array_equal(s.download(0), t.download(0))
        assert np.array_equal(s.dt_history(), t.dt_history())
