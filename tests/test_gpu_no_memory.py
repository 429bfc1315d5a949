"""A configuration whose buffers cannot be allocated (GPU): the call reports it, and
the handle works on, with the configuration before it and with that one once
memory is there.  hipMalloc is refused on the host, by a library loaded ahead of
the runtime in a process of its own."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

REFUSE = r"""
#include <dlfcn.h>
#include <stddef.h>
static int refuse;                        /* 0: none; n: the n-th hipMalloc from now */
void refuse_malloc(int n) { refuse = n; }
int hipMalloc(void **p, size_t n)
{
    static int (*real)(void **, size_t);
    if (!real) *(void **)&real = dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipMalloc");
    if (refuse && --refuse == 0) { *p = NULL; return 2; }     /* hipErrorOutOfMemory */
    return real(p, n);
}
"""

SCRIPT = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
from benchmark_spmv_using_csr_amd import _lib, matgen
from benchmark_spmv_using_csr_amd.spmv import bhsparse_spmv
A = matgen.uniform_rows(1, 20_000, 20_000, 0, 30)
x, y = matgen.vector(2, A.n), np.zeros(A.m)
op = bhsparse_spmv(np.float64)
_lib.check(op.init_platform(0), "init_platform")
_lib.check(op.set_config(0, 8, 4, 4, 0), "set_config")
_lib.check(op.prepare_mem(A.m, A.n, A.nnz, A.row_ptr, A.col, A.val, x, y), "prepare_mem")
_lib.check(op.spmv(1.0), "spmv")
_lib.check(op.get_y(), "get_y")
want = y.copy()
nth = int(sys.argv[2])
shim.refuse_malloc(nth)
try:
    rc = op.set_config(0, 4, 1, 1, 0)     # more tiles and logical waves: both buffers grow
except _lib.BhsError as e:
    rc = e.code
assert rc == _lib.BHSPARSE_OUT_OF_MEMORY, rc
shim.refuse_malloc(0)
print("refused", flush=True)
for tile in ((0, 8, 4, 4, 0), (0, 4, 1, 1, 0), (0, 8, 4, 4, 0)):
    _lib.check(op.set_config(*tile), "set_config")
    y[:] = np.nan
    _lib.check(op.spmv(1.0), "spmv")
    _lib.check(op.get_y(), "get_y")
    assert np.allclose(y, want, rtol=1e-12, atol=1e-12)
assert np.array_equal(y, want)
op.close()
print("done", flush=True)
"""


@pytest.mark.parametrize("nth", [1, 2])
def test_a_refused_allocation_leaves_the_handle_usable(nth, tmp_path):
    src, lib, script = tmp_path / "refuse.c", tmp_path / "librefuse.so", tmp_path / "script.py"
    src.write_text(REFUSE)
    script.write_text(SCRIPT)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src), "-ldl"], check=True)
    print(f"[gpu] hipMalloc number {nth} refused", flush=True)
    r = subprocess.run([sys.executable, str(script), str(lib), str(nth)], cwd=ROOT, text=True,
                       env={**os.environ, "PYTHONPATH": ROOT}, capture_output=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split() == ["refused", "done"], r.stdout + r.stderr
