"""Upload of A: a matrix large enough to be checked on the device is refused for
the same faults, with the same codes, as one checked on the host."""
import numpy as np
import pytest

from benchmark_spmv_using_csr_amd import matgen
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
