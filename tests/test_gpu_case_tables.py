"""Ybus and flows out of the case's own tables against instances that leave
them: an instance with other taps and an outage must hold the Ybus of an engine
whose case is that network (the same terms in the same order; the products of
a term may be fused differently, so 1e-14 of the largest entry), and the losses
must be the sum of the flows on either side of the branch count where their
kernel changes (1e-12 of the summed magnitudes: 1025 terms of 1.1e-16)."""
import copy

import numpy as np
import pytest

from mapol_amd.engine import CTL_OLTC, Engine
from tests.test_slot_chunks import _tree

pytestmark = pytest.mark.gpu


def _grid(n):
    case = _tree(n)
    case.Pd = np.full(n, 1e-4)
    case.B = np.full(n - 1, 1e-4)
    case.tap = np.where(np.arange(n - 1) % 3 == 0, 1.0 + 1e-3 * (np.arange(n - 1) % 7), 0.0)
    case.Gs = 1e-5 * (np.arange(n) % 5)
    return case


@pytest.mark.parametrize("n", [2, 40, 1025, 1026])
@pytest.mark.parametrize("alg", [0, 1])
def test_instances_that_leave_the_case(n, alg):
    case = _grid(n)
    m = n - 1
    taps = [b for b in range(m) if case.tap[b] != 0.0][:9]
    on = np.ones((3, m), np.uint8)
    if m > 2:
        on[1, m - 1] = 0                     # a leaf
    val = np.array([[case.tap[b] + 0.02 * t for b in taps] for t in range(3)])
    e = Engine(case, alg=alg)
    e.set_instances(br_on=on, ctl=[(CTL_OLTC, b) for b in taps], ctl_val=val)
    e.solve()
    r = e.results()
    Sf, St = e.branch_flows()
    assert (r["verdict"][[0, 2]] == 0).all()
    for t in range(3):
        c = copy.copy(case)
        c.tap = case.tap.copy()
        c.tap[taps] = val[t]
        c.br_status = on[t].copy()
        ref = Engine(c, alg=alg)
        ref.set_instances(T=1)
        ref.make_ybus()
        pairs = [(e.ybus(t), ref.ybus(0))]
        if alg and r["verdict"][t] == 0:     # the decoupled matrices too
            ref.solve()
            pairs += [(e.stage_bmat(t, w), ref.stage_bmat(0, w)) for w in (1, 2)]
        ref.close()
        for y, z in pairs:
            assert abs(y - z).max() <= 1e-14 * abs(z).max()
        if r["verdict"][t] == 0:
            s = Sf[t] + St[t]
            mag = np.abs(Sf[t]).sum() + np.abs(St[t]).sum()
            assert abs(r["loss"][t] - s.real.sum()) <= 1e-12 * mag
    e.close()
