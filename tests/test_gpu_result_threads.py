"""Results of one engine read by several host threads at once (the binding leaves
the interpreter lock during a call): flows, voltages and loadings each arrive
whole, although they leave through the engine's one set of host buffers.  The
batch is large enough for copies that are shared by threads (8 MB and more)."""
import threading

import numpy as np
import pytest

from mapol_amd import synth
from mapol_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("numbering", [0, 1])
@pytest.mark.parametrize("T", [3, 400])
def test_readers_at_once(T, numbering):
    case = synth.workload("pf1354x200", T=1)[0]
    cont = synth.n1_contingencies(case, T, 3)
    rate = np.linspace(0.5, 2.0, case.nbranch)
    e = Engine(case, bus_numbering=numbering)
    e.set_instances(br_on=cont.br_on, gen_on=cont.gen_on)
    e.solve()
    reads = [e.results, e.branch_flows, lambda: e.branch_loading(rate)]

    def arrays(x):
        return list(x.values()) if isinstance(x, dict) else list(x)

    ref = [arrays(f()) for f in reads]
    wrong = []

    def reader(k):
        for _ in range(10):
            if not all(np.array_equal(a, b) for a, b in zip(arrays(reads[k]()), ref[k])):
                wrong.append(k)

    th = [threading.Thread(target=reader, args=(k,)) for k in (0, 1, 2, 0, 1)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    e.close()
    assert not wrong
