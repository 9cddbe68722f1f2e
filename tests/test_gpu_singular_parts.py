"""A singular pivot in every place the factorization from LDS can meet it: at
level 0 (flagged by the Jacobian fill), in a part below the top (flagged to the
last launch through memory), and in the top part.  A bus whose branches are all
out has a zero row and column, so its own pivot, wherever the elimination order
puts it, is exactly zero and no other is.  Verdicts and iterations are the
oracle's, neighbouring instances stay untouched, and the next solve on the same
engine sees no flag left over."""
import numpy as np
import pytest

import oracle
from mapol_amd import synth
from mapol_amd.engine import (BPF_FDBX, BPF_FDXB, BPF_FP64, BPF_MIXED, FACTOR_LDS, SINGULAR,
                              Engine, analyse)

pytestmark = pytest.mark.gpu

DV_TOL = 1e-8


def _buses(case):
    """a load bus at elimination level 0, two at level 1 and one near the top
    whose loss leaves the rest of the grid connected"""
    import scipy.sparse as sp
    from scipy.sparse.csgraph import connected_components
    a = analyse(case)
    rp, ci, nb = a["lu_rowptr"], a["lu_colind"], a["info"]["nblocks"]
    lev = np.zeros(nb, int)
    for k in range(nb):
        up = ci[rp[k]:rp[k + 1]]
        up = up[up > k]
        if len(up):
            lev[up[0]] = max(lev[up[0]], lev[k] + 1)
    tail = set(a["tail_piv"].tolist())
    top = max(lev[k] for k in range(nb) if k not in tail)

    def alone(b):
        keep = (case.br_from != b) & (case.br_to != b)
        g = sp.coo_matrix((np.ones(keep.sum()), (case.br_from[keep], case.br_to[keep])),
                          shape=(case.nbus, case.nbus))
        return connected_components(g, directed=False)[0] == 2

    def pick(want, count):
        out = []
        for k in range(nb):
            b = int(a["bus_of_blk"][k])
            if k not in tail and want(lev[k]) and case.bus_type[b] == 1 and case.Pd[b] > 0 \
                    and case.Gs[b] == 0 and case.Bs[b] == 0 and alone(b):
                out.append(b)
            if len(out) == count:
                return out
        raise AssertionError("no such bus")

    return pick(lambda x: x == 0, 1) + pick(lambda x: x == 1, 2) + pick(lambda x: x >= top - 1, 1)


@pytest.mark.parametrize("name", ["pf1354x200", "pf9241x200"])
@pytest.mark.parametrize("kw,parts", [
    (dict(precision=BPF_MIXED), 1), (dict(precision=BPF_MIXED), 2), (dict(precision=BPF_FP64), 1),
    (dict(precision=BPF_FP64), 2), (dict(alg=BPF_FDXB), 1), (dict(alg=BPF_FDBX), 1)])
def test_singular_pivot_anywhere(name, kw, parts):
    print(f"[singular] {name} {kw} parts {parts}", flush=True)
    case, cont = synth.workload(name, T=9)
    on = cont.br_on.copy()
    bad = {}
    for t, b in zip((1, 2, 5, 7), _buses(case)):
        on[t] = (case.br_from != b) & (case.br_to != b)
        bad[t] = b
    orc = oracle.Oracle(case)
    opts = oracle.Oracle.opts(alg=kw.get("alg", 0))
    e = Engine(case, **kw)
    e.set_schedule(parts=parts)
    for masks in (on, cont.br_on, on):
        e.set_instances(br_on=masks, gen_on=cont.gen_on)
        e.solve()
        assert e.factor_form() == FACTOR_LDS
        r = e.results()
        for t in range(9):
            ro = orc.solve(opts, br_on=masks[t], gen_on=cont.gen_on[t])
            assert (r["verdict"][t] == SINGULAR) == (masks is on and t in bad), t
            assert r["verdict"][t] == ro["verdict"] and r["iterations"][t] == ro["iterations"], t
            if ro["converged"]:
                assert np.abs(r["V"][t] - ro["V"]).max() <= DV_TOL, t
    e.close()
