"""The factorization in chunks of products, which runs with the dense tail on
the vector ALUs, with other than 1024 lanes, and where the elimination tree does
not divide into parts for LDS; ``bpf_factor_form`` says which form ran.

* With 2, 4 or 8 workgroups per instance on the subtrees below the cut, or
  chosen by the active-instance count, it gives what one workgroup gives, bit
  for bit: every output keeps its product order and lane groups.
* On a grid without a plan of parts (sixty leaves on each of 45 meshed hubs: the
  leaves are one level, wider than a part, and the hubs the tail) it takes the
  tail on the matrix cores in both precisions: iterations, verdicts and voltages
  of the oracle."""
import numpy as np
import pytest

import oracle
from mapol_amd import synth
from mapol_amd.engine import (BPF_FDXB, BPF_FP64, BPF_MIXED, FACTOR_CHUNKS, FACTOR_LDS, Engine)

pytestmark = pytest.mark.gpu

DV_TOL = 1e-8
KEYS = ("V", "iterations", "verdict", "dx", "tail inverse")


def _run(case, cont, V, wg, parts, lanes, **kw):
    e = Engine(case, enforce_qlim=True, **kw)
    e.set_instances(br_on=cont.br_on, gen_on=cont.gen_on)
    e.set_factor_split(wg)
    e.set_launch(lu=lanes)
    # the forward substitution always in the factorization: whether it runs
    # there follows each part's active count and changes the rounding
    e.set_schedule(tail_inverse=2, parts=parts, fused_forward=1 << 20)
    e.solve()
    assert e.factor_form() == FACTOR_CHUNKS
    r = e.results()
    dx = e.stage_newton_step(V)
    assert e.factor_form() == FACTOR_CHUNKS
    _, Si = e.stage_tail_inverse(1)
    e.close()
    return r["V"], r["iterations"], r["verdict"], dx, Si


@pytest.mark.parametrize("name,T,lanes,kw", [
    ("pf2869x100", 12, 1024, dict(precision=BPF_MIXED, refine_steps=1)),
    ("pf9241x200", 6, 1024, dict(precision=BPF_MIXED, refine_steps=1)),
    ("pf2869x100", 8, 1024, dict(precision=BPF_FP64)),
    ("pf2869x100", 8, 512, dict(precision=BPF_FP64))])
def test_chunks_split_among_workgroups(name, T, lanes, kw):
    print(f"[forms] split {name} x {T}, {lanes} lanes, {kw}", flush=True)
    case, cont = synth.workload(name, T=T)
    rng = np.random.default_rng(11)
    V = (1 + 0.02 * rng.standard_normal((T, case.nbus))) \
        * np.exp(0.05j * rng.standard_normal((T, case.nbus)))
    base = _run(case, cont, V, 1, 1, lanes, **kw)
    for wg, parts in ((2, 1), (4, 1), (8, 1), (0, 1), (0, 4)):
        got = _run(case, cont, V, wg, parts, lanes, **kw)
        for a, b, what in zip(base, got, KEYS):
            np.testing.assert_array_equal(a, b, err_msg=f"{what}, {wg} workgroups, {parts} parts")


def _hubs(hubs=45, leaves=60):
    """meshed hubs with leaves, the hubs' loads and the leaves' in pu"""
    case = synth.workload("pf118x200", T=1)[0]
    n, h = hubs * (leaves + 1), np.arange(hubs)
    f = np.r_[h, h, np.repeat(h, leaves)]
    t = np.r_[(h + 1) % hubs, (h + 7) % hubs, np.arange(hubs, n)]
    m = len(f)
    c = {k: np.zeros(n, v.dtype) for k, v in case.__dict__.items()
         if isinstance(v, np.ndarray) and v.shape == case.Pd.shape}
    c["bus_type"] = np.ones(n, np.int32)
    c["bus_type"][0] = 3
    c["Vm"] = np.ones(n)
    c["Pd"] = np.full(n, 2e-4)
    c["Qd"] = np.full(n, 5e-5)
    for k in ("B", "tap", "shift"):
        c[k] = np.zeros(m)
    c["R"], c["X"] = np.full(m, 0.01), np.linspace(0.05, 0.1, m)
    c["br_status"] = np.ones(m, np.uint8)
    c["br_from"], c["br_to"] = f.astype(np.int32), t.astype(np.int32)
    for k in ("gen_bus", "Pg", "Qg", "Qmax", "Qmin", "VG", "gen_status"):
        c[k] = getattr(case, k)[:1].copy()
    c["gen_bus"][0] = 0
    c["VG"][0] = 1.0
    return synth.Case(**{**case.__dict__, **c, "xy": None})


@pytest.mark.parametrize("kw", [dict(precision=BPF_MIXED), dict(precision=BPF_FP64),
                                dict(precision=BPF_FP64, alg=BPF_FDXB)])
def test_grid_without_a_plan_of_parts(kw):
    print(f"[forms] hubs, {kw}", flush=True)
    case, T = _hubs(), 3
    on = np.ones((T, case.nbranch), np.uint8)
    on[1, 3] = on[2, 50] = 0               # a ring and a chord branch
    e = Engine(case, **kw)
    assert e.factor_form() == -1
    e.set_instances(br_on=on)
    e.solve()
    assert e.factor_form() == FACTOR_CHUNKS
    assert e.info()["tail_n"] >= 40
    r = e.results()
    orc = oracle.Oracle(case)
    for t in range(T):
        ro = orc.solve(oracle.Oracle.opts(alg=kw.get("alg", 0)), br_on=on[t])
        assert ro["converged"]
        assert r["verdict"][t] == ro["verdict"] and r["iterations"][t] == ro["iterations"], t
        assert np.abs(r["V"][t] - ro["V"]).max() <= DV_TOL
    e.close()


def test_form_follows_the_settings():
    case, cont = synth.workload("pf1354x200", T=4)
    e = Engine(case, precision=BPF_MIXED)
    e.set_instances(br_on=cont.br_on, gen_on=cont.gen_on)
    for kw, form in ((dict(), FACTOR_LDS), (dict(tail_inverse=2), FACTOR_CHUNKS),
                     (dict(tail_inverse=1), FACTOR_LDS)):
        e.set_schedule(**kw)
        e.solve()
        assert e.factor_form() == form
    e.adjoint()
    assert e.factor_form() == FACTOR_LDS
    e.close()
