"""Blocking calls (GPU): several threads on one handle, and the device's
scheduling flags."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from benchmark_spmv_using_csr_amd import _lib, matgen
from benchmark_spmv_using_csr_amd.spmv import bhsparse_spmv
from test_zz_no_alloc import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [500, 30_000])
def test_threads_on_one_handle(rows):
    """Every call returns success, and y is A x in the end."""
    A = matgen.uniform_rows(7, rows, rows, 1, 20)
    x = matgen.vector(8, A.n)
    op, y = bhsparse_spmv(np.float64), np.zeros(A.m)
    _lib.check(op.init_platform(0), "init_platform")
    _lib.check(op.prepare_mem(A.m, A.n, A.nnz, A.row_ptr, A.col, A.val, x, y), "prepare_mem")
    _lib.check(op.spmv(1.0), "spmv")
    _lib.check(op.get_y(), "get_y")
    want, bad = y.copy(), []

    def work():
        for _ in range(2000):
            rc = op.spmv(1.0)
            if rc:
                bad.append((rc, op._L.bhs_last_error()))

    print(f"[gpu] six threads on one handle, {rows} rows", flush=True)
    threads = [threading.Thread(target=work) for _ in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    _lib.check(op.get_y(), "get_y")
    op.close()
    assert not bad, (len(bad), bad[:3])
    assert np.array_equal(y, want)


def test_waits_sleep_where_the_device_is_set_to():
    """hipDeviceScheduleBlockingSync: a long call, and the copies behind one, leave
    the processor idle, as hipStreamSynchronize does; results are the same."""
    H = hip()
    H.hipSetDeviceFlags.argtypes = [C.c_uint]
    H.hipGetDeviceFlags.argtypes = [C.POINTER(C.c_uint)]
    A = matgen.uniform_rows(3, 400_000, 400_000, 0, 40)
    x, y, was = matgen.vector(4, A.n), np.zeros(A.m), C.c_uint()

    def handle():
        op = bhsparse_spmv(np.float64)
        _lib.check(op.init_platform(0), "init_platform")
        _lib.check(op.prepare_mem(A.m, A.n, A.nnz, A.row_ptr, A.col, A.val, x, y), "prepare_mem")
        return op

    op = handle()
    _lib.check(op.spmv(1.0), "spmv")
    _lib.check(op.get_y(), "get_y")
    op.close()
    want = y.copy()
    assert H.hipGetDeviceFlags(C.byref(was)) == 0
    assert H.hipSetDeviceFlags(4) == 0                    # hipDeviceScheduleBlockingSync
    op = handle()
    calls = {"spmv": lambda: op.spmv(1.0), "get_y": op.get_y, "set_x": lambda: op.set_x(x)}
    try:
        for name, call in calls.items():
            for _ in range(2000):                         # some 90 ms of work
                _lib.check(op.spmv_async(1.0), "spmv_async")
            w, c = time.perf_counter(), time.thread_time()
            _lib.check(call(), name)
            w, c = time.perf_counter() - w, time.thread_time() - c
            print(f"[gpu] {name}: {w * 1e3:.1f} ms, {c * 1e3:.1f} ms of processor time", flush=True)
            assert w > 0.02 and c < 0.5 * w
        _lib.check(op.spmv(1.0), "spmv")
        _lib.check(op.get_y(), "get_y")
        assert np.array_equal(y, want)
    finally:
        op.close()
        assert H.hipSetDeviceFlags(was.value) == 0
