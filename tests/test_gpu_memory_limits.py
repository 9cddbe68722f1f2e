"""Batches at the limit of the device's memory: what does not need the updates of
the factorization from LDS fits where it fitted without them.  An allocation
beside the engine leaves room for everything but them (margins of 1 GB and more
for the runtime); the solve then runs in chunks, or gives them back when a later
call needs their place, with the same results up to rounding (quadratic
convergence to 1e-8: 1e-9)."""
import contextlib
import ctypes as C

import numpy as np
import pytest

from mapol_amd import synth
from mapol_amd.engine import (BPF_FP64, BPF_MIXED, FACTOR_CHUNKS, FACTOR_LDS, Engine,
                              load_library)

pytestmark = pytest.mark.gpu


def _case(n, f, t, load):
    """a grid of load buses with the slack at bus 0"""
    case = synth.workload("pf118x200", T=1)[0]
    m = len(f)
    c = {k: np.zeros(n, v.dtype) for k, v in case.__dict__.items()
         if isinstance(v, np.ndarray) and v.shape == case.Pd.shape}
    c["bus_type"] = np.ones(n, np.int32)
    c["bus_type"][0] = 3
    c["Vm"] = np.ones(n)
    c["Pd"], c["Qd"] = np.full(n, load), np.full(n, load / 4)
    for k in ("B", "tap", "shift"):
        c[k] = np.zeros(m)
    c["R"], c["X"] = np.full(m, 0.01), np.linspace(0.05, 0.1, m)
    c["br_status"] = np.ones(m, np.uint8)
    c["br_from"], c["br_to"] = np.asarray(f, np.int32), np.asarray(t, np.int32)
    for k in ("gen_bus", "Pg", "Qg", "Qmax", "Qmin", "VG", "gen_status"):
        c[k] = getattr(case, k)[:1].copy()
    c["gen_bus"][0] = 0
    c["VG"][0] = 1.0
    return synth.Case(**{**case.__dict__, **c, "xy": None})


def _mesh(k):
    q = np.arange(k * k).reshape(k, k)
    return _case(k * k, np.r_[q[:, :-1].ravel(), q[:-1].ravel()],
                 np.r_[q[:, 1:].ravel(), q[1:].ravel()], 4e-4)


def _hip():
    """the HIP runtime that the engine's library runs on"""
    L = load_library()
    L.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    L.hipFree.argtypes = [C.c_void_p]
    L.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t)] * 2
    return L


def _free():
    L, free, total = _hip(), C.c_size_t(), C.c_size_t()
    assert L.hipDeviceSynchronize() == 0
    assert L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@contextlib.contextmanager
def _room_for(leave):
    """all of the device's free memory but `leave` bytes taken"""
    p = C.c_void_p()
    assert _hip().hipMalloc(C.byref(p), _free() - leave) == 0
    try:
        yield
    finally:
        assert _hip().hipFree(p) == 0


def _solved(case, T, precision):
    e = Engine(case, precision=precision)
    e.set_instances(T=T)
    e.solve()
    return e


@pytest.mark.parametrize("precision,T", [(BPF_FP64, 6000), (BPF_MIXED, 10000)])
def test_no_room_for_the_updates(precision, T):
    case = _mesh(40)
    free = _free()
    e = _solved(case, T, precision)
    used = free - _free()
    assert e.factor_form() == FACTOR_LDS
    i = e.info()
    lu = T * (i["nnz_lu_blocks"] + i["nblocks"]) * (32 if precision == BPF_FP64 else 16)
    ref = e.results()
    e.close()
    # the updates are more than half of the factors on a mesh: room for all the
    # rest and a quarter of the factors' size
    print(f"[memory] precision {precision}: used {used >> 20} MiB, factors {lu >> 20} MiB", flush=True)
    with _room_for(used - lu // 4):
        e = _solved(case, T, precision)
        assert e.factor_form() == FACTOR_CHUNKS
        got = e.results()
        e.close()
    for k in ("iterations", "verdict"):
        np.testing.assert_array_equal(got[k], ref[k])
    assert (ref["verdict"] == 0).all()
    assert np.abs(got["V"] - ref["V"]).max() <= 1e-9


def test_updates_given_back_for_the_adjoint():
    case, T = _mesh(40), 10000
    e = _solved(case, T, BPF_MIXED)
    assert e.factor_form() == FACTOR_LDS
    ref = e.results()
    i = e.info()
    n, m, nb, lu = case.nbus, case.nbranch, i["nblocks"], i["nnz_lu_blocks"] + i["nblocks"]
    # the adjoint's FP64 factors, tail inverses and arrays
    need = T * (32 * (lu + i["tail_n"] ** 2) + 8 * (4 * nb + 2 * n + m + 8))
    with _room_for(need - T * 16 * lu // 4):
        a = e.adjoint()
        e.solve()
        assert e.factor_form() == FACTOR_CHUNKS
        got = e.results()
    b = e.adjoint()
    e.close()
    np.testing.assert_array_equal(got["iterations"], ref["iterations"])
    assert np.abs(got["V"] - ref["V"]).max() <= 1e-9
    for k in ("grad_P", "grad_Q", "grad_x"):
        assert np.abs(a[k] - b[k]).max() <= 1e-6 * np.abs(b[k]).max(), k
