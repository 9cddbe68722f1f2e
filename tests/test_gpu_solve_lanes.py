"""The solve's lanes either side of the instance counts where the choice changes
with the buses (n / 6) and with reactive limits (3 n / 4), against 1024 lanes:
one order of sums, so the counts are equal and voltages of a quadratic
convergence agree to 1e-9."""
import numpy as np
import pytest

from mapol_amd import synth
from mapol_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,T,qlim", [
    ("pf118x200", 257, True), ("pf1354x200", 1015, True), ("pf1354x200", 1016, True),
    ("pf1354x200", 257, True), ("pf2869x100", 478, False), ("pf2869x100", 479, False)])
@pytest.mark.parametrize("precision,parts", [(0, 1), (1, 1), (1, 3)])
def test_lanes_by_buses_and_limits(name, T, qlim, precision, parts):
    case = synth.workload(name, T=1)[0]
    cont = synth.n1_contingencies(case, T, 3, gen_frac=0.25)
    out = []
    for lanes in (0, 1024):
        e = Engine(case, precision=precision, enforce_qlim=qlim)
        e.set_schedule(parts=parts)
        if lanes:
            e.set_launch(solve=lanes)
        e.set_instances(br_on=cont.br_on, gen_on=cont.gen_on)
        e.solve()
        out.append(e.results())
        e.close()
    for k in ("iterations", "verdict", "qlim_rounds"):
        np.testing.assert_array_equal(out[0][k], out[1][k])
    ok = out[1]["verdict"] == 0
    assert ok.sum() > T // 2
    assert np.abs(out[0]["V"][ok] - out[1]["V"][ok]).max() <= 1e-9
