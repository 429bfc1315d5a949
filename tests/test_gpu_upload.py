"""Copies between host and device: a matrix large enough to be checked on the
device is refused for the same faults, with the same codes, as one checked on the
host; x and y arrive whole by every route (staged or not, several threads)."""
import threading

import numpy as np
import pytest

from benchmark_spmv_using_csr_amd import batched, matgen
from benchmark_spmv_using_csr_amd._lib import (BHSPARSE_INVALID_MATRIX, BHSPARSE_NOT_INITIALIZED,
                                               spmv_lib)
from benchmark_spmv_using_csr_amd.spmv import bhsparse_spmv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [3000, 40_000])     # 51,000 and 680,000 entries
@pytest.mark.parametrize("what", ["row_first", "row_last", "col_first", "col_mid", "col_last",
                                  "col_negative"])
@pytest.mark.parametrize("loaded", [False, True])
def test_a_bad_matrix_is_refused(rows, what, loaded):
    A = matgen.uniform_rows(3, rows, rows, 16, 16)
    assert A.nnz == 16 * rows
    nnz = A.nnz - 1                                  # a remainder of three indices
    rp, col, val = A.row_ptr.copy(), A.col[:-1].copy(), A.val[:-1].copy()
    rp[-1] -= 1
    x, y = matgen.vector(4, A.n), np.zeros(A.m)
    good_rp, good_col = rp.copy(), col.copy()
    if what == "row_first":
        rp[1], rp[2] = rp[2] + 1, rp[1]
    elif what == "row_last":
        rp[-2] = rp[-1] + 1
    else:
        at = {"col_first": 0, "col_mid": nnz // 2 + 1, "col_last": nnz - 1,
              "col_negative": nnz - 3}[what]
        col[at] = -1 if what == "col_negative" else A.n
    op = bhsparse_spmv(np.float64)

    def prepare(r, c):
        return op.prepare_mem(A.m, A.n, nnz, r, c, val, x, y)

    try:
        assert op.init_platform(0) == 0
        if loaded:
            assert prepare(good_rp, good_col) == 0
        assert prepare(rp, col) == BHSPARSE_INVALID_MATRIX
        msg = spmv_lib().bhs_last_error().decode()
        assert msg == ("row_ptr is not monotone" if what.startswith("row")
                       else "column index out of range")
        if not loaded:
            assert op.spmv(1.0) == BHSPARSE_NOT_INITIALIZED
            assert prepare(good_rp, good_col) == 0
        assert op.spmv(1.0) == 0 and op.get_y() == 0
        want = np.add.reduceat(val * x[good_col], good_rp[:-1])
        scale = np.add.reduceat(np.abs(val * x[good_col]), good_rp[:-1])
        assert np.all(np.abs(y - want) <= 32 * np.finfo(np.float64).eps * scale)
    finally:
        op.close()


def _identity(n):
    return matgen.CSR(n, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32),
                      np.ones(n))


def _round_trips(n, dtype, seed, times):
    """x through set_x, a diagonal matrix and get_y: exact, by value."""
    A, rng = _identity(n), np.random.default_rng(seed)
    op = bhsparse_spmv(dtype)
    try:
        assert op.init_platform(0) == 0
        y = np.zeros(n + 3, dtype)                   # three guards behind y
        y[n:] = 7
        x = rng.random(n).astype(dtype)
        assert op.prepare_mem(n, n, n, A.row_ptr, A.col, A.val.astype(dtype), x, y) == 0
        assert op.spmv(1.0) == 0 and op.get_y() == 0
        ok = np.array_equal(y[:n], x)
        for _ in range(times):
            x = rng.random(n).astype(dtype)
            assert op.set_x(x) == 0
            x2 = x.copy()
            x[:] = 0                                 # the call has read x when it returns
            assert op.spmv(1.0) == 0 and op.get_y() == 0
            ok = ok and np.array_equal(y[:n], x2)
        return ok and bool(np.all(y[n:] == 7))
    finally:
        op.close()


# 16 KB pieces, chunks of 256 KB and 1 MB, the two halves of 2 MB, the reuse of the ring
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("words", [2, 6, 1022, 4094, 4096, 4098, 8200, 32766, 65534, 65536,
                                   65538, 262146, 524286, 524290, 1048578, 2097152, 2097154, 5000002])
def test_x_and_y_arrive(words, dtype):
    assert _round_trips(words // (np.dtype(dtype).itemsize // 4), dtype, words, 3)


def test_x_and_y_arrive_in_threads():
    """More threads than pinned buffers, both directions."""
    sizes = [33, 4000, 16_000, 300_000, 700_001, 5]
    out = [None] * len(sizes)

    def work(i):
        out[i] = _round_trips(sizes[i], np.float64, i, 20)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert out == [True] * len(sizes)


@pytest.mark.parametrize("sizes", [[1, 40, 0, 7], [3000, 17_000, 64], [9000] * 40, [300_000, 5, 90_001]])
def test_batch_x_and_y_arrive(sizes):
    rng = np.random.default_rng(len(sizes))
    ks = [(1, 4, 16, 3)[i % 4] for i in range(len(sizes))]
    b = batched.SpmvBatch([_identity(n) for n in sizes], ks, np.float64)
    try:
        for _ in range(3):
            X = [rng.random((n, k)) for n, k in zip(sizes, ks)]
            b.set_x(X)
            b.run(1.0)
            assert all(np.array_equal(g, x) for g, x in zip(b.y(), X))
            b.run_plain(1.0)
            assert all(np.array_equal(g, x) for g, x in zip(b.y(plain=True), X))
    finally:
        b.close()


def test_more_handles_than_signal_words():
    """258 open handles: the last ones wait by synchronising their stream."""
    A = _identity(10)
    ops, ys = [], []
    try:
        for i in range(258):
            op = bhsparse_spmv(np.float64)
            ops.append(op)
            ys.append(np.zeros(10))
            assert op.init_platform(0) == 0
            x = np.arange(10) + i + 1.0
            assert op.prepare_mem(10, 10, 10, A.row_ptr, A.col, A.val, x, ys[-1]) == 0
        for _ in range(2):
            for i, op in enumerate(ops):
                assert op.spmv(2.0) == 0 and op.get_y() == 0
                assert np.array_equal(ys[i], 2 * (np.arange(10) + i + 1.0))
    finally:
        for op in ops:
            op.close()
