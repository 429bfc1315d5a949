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
