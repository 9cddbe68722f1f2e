"""Batches whose instances x branches exceed the 2^32 threads of a launch, which
the runtime would cut short without an error: the Ybus positions of changed
branches (a thread per position of 17 000 branches x 65 528 instances is 4.46e9)
and the branch flows (66 000 x 65 528 is 4.32e9; 190 GB of the device).  The grid
is one of parallel branches; a few instances spread over the batch have another
tap.  Their Ybus holds the sum of the branches with that tap (numpy; 1e-12 of
the entries), and voltages and losses are those of the same instances in
a small batch (the same sums; the losses in another order, 1e-12 of the summed
flows)."""
import numpy as np
import pytest

from mapol_amd.engine import CTL_OLTC, Engine
from tests.test_gpu_memory_limits import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(2, 17000), (140, 66000)])
def test_more_branches_than_threads_of_a_launch(n, m):
    T = 65528
    f = np.arange(m) % (n - 1)
    par = m // (n - 1)               # branches side by side
    case = _case(n, f, f + 1, 0.01 / n)     # (0.1 / n has no solution on the chain)
    case.R, case.X = case.R * par, case.X * par
    k = m // 3
    case.tap[k] = 1.0                # a tap changer, which the control sets
    val = np.full((T, 1), np.nan)
    at = np.array([0, 1, 7, 8, 32771, T - 9, T - 1])
    val[at, 0] = 1.0 + 0.01 * (1 + np.arange(len(at)))

    def solve(v, which):
        print(f"[grid] {n} buses, {m} branches x {len(v)}", flush=True)
        e = Engine(case, maxit_nr=10)
        e.set_instances(T=len(v), ctl=[(CTL_OLTC, k)], ctl_val=v)
        e.solve()
        r = e.results()
        y = [e.ybus(t) for t in which]
        e.close()
        return r, y

    r, y = solve(val, at)
    s, z = solve(val[at], range(len(at)))
    assert (r["verdict"] == 0).all()
    same = np.setdiff1d(np.arange(T), at)
    assert (r["loss"][same] == r["loss"][same[0]]).all()
    assert len(set(r["loss"][at])) == len(at) and r["loss"][same[0]] not in r["loss"][at]
    a, b = case.br_from[k], case.br_to[k]
    pair = case.br_from == a
    ys = 1.0 / (case.R + 1j * case.X)
    for q, t in enumerate(at):
        ft = -(ys[pair].sum() + ys[k] / val[t, 0] - ys[k])
        for got in (y[q], z[q]):
            assert abs(got[a, b] - ft) <= 1e-12 * abs(ft)
        assert abs(y[q] - z[q]).max() <= 1e-12 * abs(z[q]).max()
        assert np.abs(r["V"][t] - s["V"][q]).max() <= 1e-12
        # a pair of buses carries at most the whole load, 0.01 pu, and its losses
        assert abs(r["loss"][t] - s["loss"][q]) <= 1e-12 * 0.02 * (n - 1)
