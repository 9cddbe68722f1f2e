"""The loading report's device buffer: kept between calls for ordinary batches,
given back after the call for large ones (2000 parallel branches x 5000
instances: 80 MB of loadings, in the caller's numbering)."""
import numpy as np
import pytest

from mapol_amd.engine import Engine
from tests.test_gpu_memory_limits import _case, _free

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,kept", [(5000, False), (500, True)])
def test_loading_buffer(T, kept):
    m = 2000
    case = _case(2, np.zeros(m), np.ones(m), 0.1)
    case.R, case.X = case.R * m, case.X * m
    e = Engine(case, bus_numbering=0)
    e.set_instances(T=T)
    e.solve()
    rate = np.full(m, 1e-3)
    small = e.branch_loading_noalloc(rate)     # takes no device memory
    e.branch_flows()
    before = _free()
    a = e.branch_loading(rate)
    e.branch_flows()             # the runtime lets go of a freed buffer with the next copy
    held = before - _free()
    b = e.branch_loading(rate)
    e.close()
    for k in a:
        np.testing.assert_array_equal(a[k], b[k])
        np.testing.assert_array_equal(a[k], small[k])
    # the rows alone are 8 T m bytes
    assert (held >= 8 * T * m) if kept else (held < 8 * T * m // 2), held
