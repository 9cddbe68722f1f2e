"""The dense tail's inverse at the sizes where its quad and tile edges fall:
one pivot, odd and even counts, either side of a 16-row strip (8 pivots), a
32-row tile (16), three tiles (48) and the whole matrix, in both precisions,
against numpy's inverse of the oracle's Schur complement.  Tolerance: the
forward error of an inverse without pivoting, 8 n eps cond(S) of the largest
entry for n scalars (the factorization below the tail included)."""
import numpy as np
import pytest

import oracle
from mapol_amd import synth
from mapol_amd.engine import Engine
from tests.test_gpu_stages import _superset_jacobian

pytestmark = pytest.mark.gpu

LIMITS = (1, 2, 3, 8, 9, 15, 16, 17, 31, 33, 47, 48, 49, 57, 64)


@pytest.mark.parametrize("prec", [0, 1])
def test_tail_inverse_at_every_edge(prec):
    case, cont = synth.workload("pf118x200", T=2)
    orc = oracle.Oracle(case)
    sizes = set()
    for limit in LIMITS:
        print(f"[tail quads] precision {prec} limit {limit}", flush=True)
        e = Engine(case, precision=prec, tail_limit=limit)
        e.set_instances(br_on=cont.br_on, gen_on=cont.gen_on)
        e.solve()
        r = e.results()
        V = r["V"] * (1 + 1e-3 * np.random.default_rng(5).normal(size=r["V"].shape))
        e.stage_newton_step(V)
        for t in range(2):
            bus, Si = e.stage_tail_inverse(t)
            s = len(bus)
            sizes.add(s)
            if s == 0:                  # the limit holds no whole level
                continue
            J, blk = _superset_jacobian(
                case, orc.jacobian(V[t], br_on=cont.br_on[t], gen_on=cont.gen_on[t]),
                r["bus_type"][t])
            J = J.toarray()
            at = np.array([2 * blk[int(b)] + q for b in bus for q in (0, 1)])
            rest = np.setdiff1d(np.arange(len(J)), at)
            S = J[np.ix_(at, at)] - J[np.ix_(at, rest)] @ np.linalg.solve(
                J[np.ix_(rest, rest)], J[np.ix_(rest, at)])
            ref = np.linalg.inv(S)
            eps = np.finfo(np.float64 if prec == 0 else np.float32).eps
            err = np.abs(Si - ref).max() / np.abs(ref).max()
            assert err <= 8 * 2 * s * eps * np.linalg.cond(S), (limit, s, t, err)
        e.close()
    # the engine takes whole levels, and none below four of them
    assert min(sizes - {0}) <= 8 and max(sizes) >= 48 and any(s % 2 for s in sizes), sizes
