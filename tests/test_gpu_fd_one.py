"""The decoupled loop in one launch against its launches per half-step (which
per-kernel timing takes), either side of the rule's edges, with iteration caps
that end some instances early and with an instance that starts non-finite.
The arithmetic is the same up to the fusing of products: voltages within 1e-9
(the loop ends at a mismatch of 1e-8 and contracts linearly), counts equal."""
import numpy as np
import pytest

from mapol_amd import synth
from mapol_amd.engine import BPF_FDBX, BPF_FDXB, CTL_AVR, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,T", [("pf118x200", 1), ("pf118x200", 1024), ("pf118x200", 1025),
                                    ("pf1354x200", 3), ("pf2869x100", 2), ("pf9241x200", 2)])
@pytest.mark.parametrize("alg,maxit", [(BPF_FDXB, 30), (BPF_FDBX, 30), (BPF_FDXB, 1),
                                       (BPF_FDXB, 5)])
def test_one_launch_matches_half_steps(name, T, alg, maxit):
    case, cont = synth.workload(name, T=T)
    e = Engine(case, alg=alg, maxit_fd=maxit)
    pv = int(np.flatnonzero(np.asarray(case.bus_type) == 2)[0])
    val = np.full((T, 1), np.nan)
    if T > 1:
        val[T - 1] = np.inf
    e.set_instances(br_on=cont.br_on, gen_on=cont.gen_on, ctl=[(CTL_AVR, pv)], ctl_val=val)
    e.solve()
    one = e.results()
    e.set_timing(True)
    e.solve()
    ref = e.results()
    e.close()
    for k in ("iterations", "verdict", "bus_type"):
        np.testing.assert_array_equal(one[k], ref[k])
    ok = np.isfinite(ref["norm"]) & np.isfinite(ref["V"]).all(axis=1)
    assert ok.sum() >= max(1, T - 1)
    assert np.abs(one["V"][ok] - ref["V"][ok]).max() <= 1e-9
    if T > 1:
        assert one["verdict"][T - 1] == 3
