"""Which kernels a handle's call enqueues (GPU): the choice follows from the
matrix and the configuration in force, not from the configurations before it."""
import ctypes as C

import numpy as np
import pytest

from benchmark_spmv_using_csr_amd import _lib, matgen
from benchmark_spmv_using_csr_amd.spmv import bhsparse_spmv
from test_zz_no_alloc import hip

pytestmark = pytest.mark.gpu


def kernels_of_a_call(op):
    """Number of nodes that spmv_async leaves in a captured graph."""
    H, st = hip(), C.c_void_p()
    _lib.check(op._fn("get_stream")(op._h, C.byref(st)), "get_stream")
    graph, n = C.c_void_p(), C.c_size_t()
    H.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    H.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    H.hipGraphGetNodes.argtypes = [C.c_void_p, C.c_void_p, C.POINTER(C.c_size_t)]
    H.hipGraphDestroy.argtypes = [C.c_void_p]
    assert H.hipStreamBeginCapture(st, 0) == 0
    rc = op.spmv_async(1.0)
    assert H.hipStreamEndCapture(st, C.byref(graph)) == 0
    _lib.check(rc, "spmv_async")
    assert H.hipGraphGetNodes(graph, None, C.byref(n)) == 0
    assert H.hipGraphDestroy(graph) == 0
    return n.value


def loaded(A, dtype):
    op, y = bhsparse_spmv(dtype), np.full(A.m, np.nan, dtype)
    _lib.check(op.init_platform(0), "init_platform")
    _lib.check(op.prepare_mem(A.m, A.n, A.nnz, A.row_ptr, A.col, A.val.astype(dtype),
                              matgen.vector(6, A.n).astype(dtype), y), "prepare_mem")
    return op, y


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("waves", [1, 4])
def test_a_plain_class_after_csr_vector(dtype, waves):
    """csr-vector's classes share a plain class's tile; the plain kernel is chosen
    as on a fresh handle, and y is the same bits."""
    A = matgen.uniform_rows(5, 40_000, 40_000, 0, 30)
    plain, vector = (0, 8, waves, 1, 0), (1, 8, 4, 1, 8)
    op, y = loaded(A, dtype)
    _lib.check(op.set_config(*plain), "set_config")
    want = kernels_of_a_call(op)
    _lib.check(op.spmv(0.5), "spmv")
    _lib.check(op.get_y(), "get_y")
    fresh = y.copy()
    op.close()
    op, y = loaded(A, dtype)
    for _ in range(2):
        _lib.check(op.set_config(*vector), "set_config")
        assert kernels_of_a_call(op) == 1
        _lib.check(op.set_config(*plain), "set_config")
        print(f"[gpu] plain after csr-vector, {np.dtype(dtype).name}, {waves} waves", flush=True)
        assert kernels_of_a_call(op) == want == 1
        _lib.check(op.spmv(0.5), "spmv")
        _lib.check(op.get_y(), "get_y")
        assert np.array_equal(y, fresh)
    op.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_long_rows_on_average_leave_the_fused_kernel(dtype):
    """The line lies at a mean row of one logical wave: at T = 1 the loop and a
    calibration beyond it, at T = 4 from 1,024 logical waves on; y is the same bits
    on both sides (one empty row more or less does not move a sum)."""
    rng = np.random.default_rng(2)
    for tile, length, rows, beyond in [((0, 8, 4, 1, 0), 512, 700, 2),
                                       ((0, 8, 4, 4, 0), 2048, 300, 1),
                                       ((0, 8, 4, 4, 0), 2048, 1100, 2)]:
        nnz, n = length * rows, 50_000
        cuts = np.sort(rng.choice(nnz, rows - 2, False))         # rows - 1 rows of any length
        row_ptr = np.r_[0, cuts, nnz].astype(np.int32)
        col, val = rng.integers(0, n, nnz).astype(np.int32), rng.uniform(-1, 1, nnz).astype(dtype)
        x, got = rng.uniform(-1, 1, n).astype(dtype), []
        for extra, kernels in ((0, beyond), (1, 1)):             # rows - 1, then rows of them
            rp = np.r_[row_ptr, np.full(extra, nnz, np.int32)].astype(np.int32)
            op, y = bhsparse_spmv(dtype), np.full(len(rp) - 1, np.nan, dtype)
            _lib.check(op.init_platform(0), "init_platform")
            _lib.check(op.set_config(*tile), "set_config")
            _lib.check(op.prepare_mem(len(rp) - 1, n, nnz, rp, col, val, x, y), "prepare_mem")
            print(f"[gpu] {tile} {rows - 1 + extra} rows, {nnz} nonzeros", flush=True)
            assert kernels_of_a_call(op) == kernels
            for _ in range(2):
                _lib.check(op.spmv(1.0), "spmv")
            _lib.check(op.get_y(), "get_y")
            op.close()
            got.append(y[:rows - 1])
        assert np.array_equal(*got)
