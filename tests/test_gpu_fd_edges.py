"""The decoupled loop in one launch or by half-steps, either side of the bus and
instance counts where the choice changes (64 and 65 buses at 6 and 3 instances
per compute unit, 699 and 700, 2500 and 2501 at a quarter, 3000 and 3001),
against the half-steps, which per-kernel timing takes.  The arithmetic is the
same up to the fusing of products: voltages within 1e-9 (the loop ends at a
mismatch of 1e-8 and contracts linearly), counts equal."""
import numpy as np
import pytest

from mapol_amd import synth
from mapol_amd.engine import BPF_FDBX, BPF_FDXB, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,T", [(64, 1536), (64, 1537), (65, 768), (65, 769), (699, 769),
                                 (700, 769), (2500, 63), (2501, 63), (2501, 64), (3000, 64),
                                 (3001, 64)])
@pytest.mark.parametrize("alg", [BPF_FDXB, BPF_FDBX])
def test_either_side_of_the_rule(n, T, alg):
    for seed in range(5, 12):
        try:
            case = synth.make_grid(n, n // 6, int(1.6 * n), seed, load_scale=0.2, start="solved")
            break
        except RuntimeError:                 # this seed's base case has no solution
            continue
    cont = synth.n1_contingencies(case, T, 3)
    e = Engine(case, alg=alg)
    e.set_instances(br_on=cont.br_on, gen_on=cont.gen_on)
    e.solve()
    one = e.results()
    e.set_timing(True)
    e.solve()
    ref = e.results()
    e.close()
    for k in ("iterations", "verdict"):
        np.testing.assert_array_equal(one[k], ref[k])
    ok = ref["verdict"] == 0
    assert ok.sum() > 0.9 * T
    assert np.abs(one["V"][ok] - ref["V"][ok]).max() <= 1e-9
