"""Results on their way to the host at the sizes where the way changes: one
gathering kernel up to 2 MB, one copying thread up to 8 MB, four beyond, chunks
of 1 MB; in both bus numberings.  Instances repeat seven outages, so every row
must be the row of the seven-instance batch (which takes the first way).
Tolerance 1e-9: the batch size may choose another summation order in the
factorization of converged (1e-8) systems with quadratic convergence; two rows
that change places differ by 1e-3 and more."""
import numpy as np
import pytest

from mapol_amd import synth
from mapol_amd.engine import Engine

pytestmark = pytest.mark.gpu

N, M = 118, 186                      # buses and branches of the case
SMALL = (2 << 20) // (17 * N + 40)   # the largest batch of the first way
SPLIT_V = (8 << 20) // (16 * N)      # one thread for the voltages
SPLIT_L = (8 << 20) // (8 * M)       # one thread for the loadings


@pytest.mark.parametrize("numbering", [0, 1])
@pytest.mark.parametrize("T", [1, SMALL, SMALL + 1, SPLIT_V, SPLIT_V + 1, SPLIT_L + 1])
def test_rows_arrive_where_they_belong(T, numbering):
    case, cont = synth.workload("pf118x200", T=7)
    assert (case.nbus, case.nbranch) == (N, M)
    rate = np.linspace(0.2, 2.0, M)

    def solve(t):
        e = Engine(case, bus_numbering=numbering)
        k = np.arange(t) % 7
        e.set_instances(br_on=cont.br_on[k], gen_on=cont.gen_on[k])
        e.solve()
        out = e.results(), e.branch_loading(rate), e.adjoint(rate=rate, w=1.0), \
            e.branch_loading_noalloc(rate), e.branch_flows()
        e.close()
        return out

    ref_r, ref_l, ref_a, _, ref_f = solve(7)
    r, l, a, same, f = solve(T)
    k = np.arange(T) % 7
    for x, y in ((r["V"], ref_r["V"]), (r["loss"], ref_r["loss"]), (f[0], ref_f[0]),
                 (f[1], ref_f[1]), (l["loading"], ref_l["loading"]),
                 (a["grad_P"], ref_a["grad_P"]), (a["grad_x"], ref_a["grad_x"])):
        assert np.abs(x - y[k]).max() <= 1e-9 * max(1.0, np.abs(y).max())
    for key in ("iterations", "verdict", "qlim_rounds", "bus_type"):
        np.testing.assert_array_equal(r[key], ref_r[key][k])
    np.testing.assert_array_equal(l["overloads"], ref_l["overloads"][k])
    for key in ("loading", "overloads", "max_loading"):
        np.testing.assert_array_equal(l[key], same[key])
