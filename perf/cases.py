"""What is timed of the CSR SpMV library: one dict of plain values per case.

Five kinds of pass, each through the public entry points:

* ``device``: y = alpha A x over the caller's own device arrays
  (``bhs_{s,d}_spmv_noalloc`` on torch tensors and torch's current stream), as a
  solver calls it that keeps its vectors on the GPU.
* ``loop``: a handle with A and x loaded, ``runs`` SpMVs in a row and then
  ``get_y``: the reference driver's protocol (NUM_RUN calls of run_benchmark(),
  spmv_cuda/main.cu:808-821).
* ``host``: a handle whose caller keeps its vectors on the host, as the
  reference's interface has it: ``set_x``, ``spmv``, ``get_y``.
* ``once``: the reference driver's whole sequence for one matrix on an
  initialised platform: ``prepare_mem``, ``run_benchmark``, ``get_y``,
  ``free_mem`` (main.cu:772-825).
* ``batch``: a batch of matrices with 1, 4 or 16 right-hand sides each, given
  new right-hand sides: ``set_x``, ``run``, ``y``.

Matrices come from the package's seeded generators: rows of uniform length,
power-law rows, bands, the 7-point Laplacian and 3x3 blocks.
"""
from __future__ import annotations

import numpy as np
import torch

from benchmark_spmv_using_csr_amd import _lib, batched, matgen, tuner
from benchmark_spmv_using_csr_amd.spmv import bhsparse_spmv

MAX_NNZ = 54_000_000      # the largest matrix of the list (3x3 blocks)
LOOP_NNZ = 10_000_000     # the largest matrix of a loop
HOST_NNZ = 10_000_000     # the largest of the passes that copy on each call


def listed():
    return [
        # a coarse grid or a test problem: what a call costs by itself
        dict(name="device_tiny_f64", kind="device", family="uniform", m=1000, n=1000, longest=16,
             dtype="float64", alpha=1.0),
        # the benchmark's 65,536-row matrix of short uniform rows, single precision
        dict(name="device_uniform_65536_f32", kind="device", family="uniform", m=65536, n=65536,
             longest=32, dtype="float32", alpha=1.0),
        # a rectangular matrix with ragged rows and a partial last tile
        dict(name="device_powerlaw_rect_f64", kind="device", family="powerlaw", m=200_000,
             n=180_000, exponent=2.0, longest=50_000, empty=0.1, nnz=2_000_003, dtype="float64",
             alpha=-0.75),
        # the headline matrix (a graph with power-law degrees), in a device-side
        # solver such as a power iteration
        dict(name="device_powerlaw_1m_f64", kind="device", family="powerlaw", m=1 << 20,
             n=1 << 20, exponent=2.0, longest=100_000, empty=0.1, nnz=10_000_000,
             dtype="float64", alpha=1.0),
        # a Krylov step on the 7-point stencil
        dict(name="device_laplace_160_f64", kind="device", family="laplace", m=160 ** 3,
             n=160 ** 3, side=160, dtype="float64", alpha=1.0),
        # a finite-element matrix of 3x3 blocks, the largest, single precision
        dict(name="device_block3_2m_f32", kind="device", family="block3", m=2_000_000,
             n=2_000_000, bandwidth=5000, dtype="float32", alpha=1.0),
        # the reference driver's timed loop on the headline matrix, tile from the tuner
        dict(name="loop_powerlaw_1m_f64", kind="loop", family="powerlaw", m=1 << 20, n=1 << 20,
             exponent=2.0, longest=100_000, empty=0.1, nnz=10_000_000, dtype="float64",
             alpha=1.0, runs=200, tuned=True, wait=True),
        # the same on the 65,536-row matrix, where launch and waiting count
        dict(name="loop_uniform_65536_f64", kind="loop", family="uniform", m=65536, n=65536,
             longest=32, dtype="float64", alpha=1.0, runs=200, tuned=True, wait=True),
        # a band of odd size at the default tile, calls enqueued without waiting
        dict(name="loop_banded_f32", kind="loop", family="banded", m=300_001, n=300_001,
             bandwidth=27, dtype="float32", alpha=1.0, runs=200, tuned=False, wait=False),
        # an iterative solver with its vectors on the host
        dict(name="host_laplace_100_f64", kind="host", family="laplace", m=100 ** 3, n=100 ** 3,
             side=100, dtype="float64", alpha=1.0, tuned=True),
        # one matrix from host CSR to host y
        dict(name="once_powerlaw_1m_f64", kind="once", family="powerlaw", m=1 << 20, n=1 << 20,
             exponent=2.0, longest=100_000, empty=0.1, nnz=10_000_000, dtype="float64",
             alpha=1.0),
        # many systems with several right-hand sides each
        dict(name="batch_24_f64", kind="batch", mats=24, m_lo=1000, m_hi=100_000,
             dtype="float64", alpha=1.0),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _family(rng, most):
    """A matrix of at most about `most` nonzeros: sizes log-uniform, odd ones among them."""
    f = rng.choice(["uniform", "powerlaw", "banded", "laplace", "block3"])
    if f == "laplace":
        side = _log(rng, 10, min(160, int((most / 7) ** (1 / 3))))
        return dict(family=f, m=side ** 3, n=side ** 3, side=side)
    if f == "uniform":
        longest = rng.randint(4, 64)
        m = _log(rng, 1000, min(2_000_000, 2 * most // longest))
        return dict(family=f, m=m, n=max(longest, int(m * rng.uniform(0.5, 2.0))),
                    longest=longest)
    if f == "banded":
        bw = rng.randint(1, 100) * 2 + 1
        m = _log(rng, 1000, min(2_000_000, most // bw))
        return dict(family=f, m=m, n=m, bandwidth=bw)
    if f == "block3":
        m = _log(rng, 1000, min(2_000_000, most // 27))
        return dict(family=f, m=m, n=m, bandwidth=rng.randint(30, 5000))
    m = _log(rng, 1000, min(1 << 20, most // 9))
    return dict(family=f, m=m, n=m, exponent=round(rng.uniform(1.8, 3.0), 3),
                longest=min(100_000, m), empty=round(rng.uniform(0.0, 0.2), 3),
                nnz=_log(rng, m, min(most, 16 * m)))


def draw(rng):
    kind = rng.choice(["device"] * 5 + ["loop"] * 3 + ["host", "once", "batch"])
    dtype = rng.choice(["float64", "float32"])
    alpha = rng.choice([1.0, 1.0, round(rng.uniform(-2.0, 2.0), 3)])
    if kind == "batch":
        lo = _log(rng, 100, 4000)
        return dict(kind=kind, mats=rng.randint(4, 24), m_lo=lo, m_hi=lo * rng.randint(4, 24),
                    dtype=dtype, alpha=alpha)
    case = dict(kind=kind, dtype=dtype, alpha=alpha)
    if kind == "device":
        return {**case, **_family(rng, MAX_NNZ)}
    if kind == "loop":
        return {**case, **_family(rng, LOOP_NNZ), "runs": 200, "tuned": rng.random() < 0.6,
                "wait": rng.random() < 0.5}
    if kind == "host":
        case["tuned"] = rng.random() < 0.6
    return {**case, **_family(rng, HOST_NNZ)}


def _matrix(case, seed):
    """The case's CSR (values in the case's type) and x, from the seed."""
    f, m, n = case["family"], case["m"], case["n"]
    if f == "uniform":
        A = matgen.uniform_rows(seed, m, n, 0, case["longest"])
    elif f == "powerlaw":
        A = matgen.power_law(seed, m, n, case["exponent"], case["longest"], case["empty"],
                             case["nnz"])
    elif f == "banded":
        A = matgen.banded(seed, m, n, case["bandwidth"])
    elif f == "laplace":
        A = matgen.laplacian7(case["side"], case["side"], case["side"])
    else:
        A = matgen.block3(seed, m, 9, case["bandwidth"])
    dtype = np.dtype(case["dtype"])
    return A.astype(dtype), matgen.vector(seed + 7919, n).astype(dtype)


def _batch_sizes(case):
    """(m, k, family, parameter) of every matrix of a batch: the four families of
    batched.batch_set, m log-uniform, k in {1, 4, 16}; the same for every seed."""
    rng = np.random.default_rng([case["mats"], case["m_lo"], case["m_hi"]])
    sizes = []
    for i in range(case["mats"]):
        m = int(case["m_lo"] * (case["m_hi"] / case["m_lo"]) ** rng.random())
        k = int(rng.choice([1, 4, 16]))
        f = ("uniform", "powerlaw", "banded", "block3")[i % 4]
        p = (int(rng.integers(4, 65)) if f == "uniform" else
             float(rng.uniform(1.5, 3.0)) if f == "powerlaw" else
             int(rng.integers(1, 101)) * 2 + 1 if f == "banded" else int(rng.integers(30, 5001)))
        sizes.append((m, k, f, p))
    return sizes


def _batch(case, seed):
    dtype = np.dtype(case["dtype"])
    mats, ks, Xs = [], [], []
    for i, (m, k, f, p) in enumerate(_batch_sizes(case)):
        s = seed * 1000 + i
        A = (matgen.uniform_rows(s, m, m, 0, p) if f == "uniform" else
             matgen.power_law(s, m, m, p, min(100_000, m), 0.1, 0) if f == "powerlaw" else
             matgen.banded(s, m, m, p) if f == "banded" else matgen.block3(s, m, 9, p))
        mats.append(A.astype(dtype))
        ks.append(k)
        Xs.append(matgen.vector(s + 7919, m * k).reshape(m, k).astype(dtype))
    return mats, ks, Xs


def _handle(case, A, x):
    op = bhsparse_spmv(A.val.dtype)
    _lib.check(op.init_platform(0), "init_platform")
    y = np.zeros(A.m, A.val.dtype)
    if case["kind"] != "once":
        _lib.check(op.prepare_mem(A.m, A.n, A.nnz, A.row_ptr, A.col, A.val, x, y), "prepare_mem")
        if case["tuned"]:
            net = tuner.make_net(tuner.load_net())
            op.apply_tuner(net, tuner.CLASSES)
            net.close()
    return op, y


def prepare(case, seed):
    state = dict(case=case)
    if case["kind"] == "batch":
        mats, ks, Xs = _batch(case, seed)
        state.update(op=batched.SpmvBatch(mats, ks, np.dtype(case["dtype"])), Xs=Xs)
        return state
    A, x = _matrix(case, seed)
    if case["kind"] == "device":
        L = _lib.spmv_lib()
        state["call"] = (L.bhs_d_spmv_noalloc if case["dtype"] == "float64"
                         else L.bhs_s_spmv_noalloc)
        state["size"] = (A.m, A.n, A.nnz)
        state["arrays"] = [torch.from_numpy(a).cuda() for a in (A.row_ptr, A.col, A.val, x)]
        state["y"] = torch.empty(A.m, dtype=state["arrays"][3].dtype, device="cuda")
        return state
    op, y = _handle(case, A, x)
    state.update(op=op, x=x, y=y)
    if case["kind"] == "once":
        state["A"] = A
    return state


def run(state):
    case, check = state["case"], _lib.check
    kind, alpha = case["kind"], case["alpha"]
    if kind == "device":
        row_ptr, col, val, x = state["arrays"]
        y = state["y"]
        check(state["call"](*state["size"], row_ptr.data_ptr(), col.data_ptr(), val.data_ptr(),
                            x.data_ptr(), y.data_ptr(), alpha,
                            torch.cuda.current_stream().cuda_stream), "spmv_noalloc")
        return y
    op = state["op"]
    if kind == "batch":
        op.set_x(state["Xs"])
        op.run(alpha)
        return op.y()
    if kind == "loop":
        call = op.spmv if case["wait"] else op.spmv_async
        for _ in range(case["runs"]):
            check(call(alpha), "spmv")
    elif kind == "host":
        check(op.set_x(state["x"]), "set_x")
        check(op.spmv(alpha), "spmv")
    else:
        A = state["A"]
        check(op.prepare_mem(A.m, A.n, A.nnz, A.row_ptr, A.col, A.val, state["x"], state["y"]),
              "prepare_mem")
        check(op.spmv(alpha), "spmv")
    check(op.get_y(), "get_y")
    if kind == "once":
        check(op.free_mem(), "free_mem")
    return state["y"]


def _count(case):
    """(m, n, nnz) of the case's matrix: nnz as its generator draws it (its mean)."""
    f, m, n = case["family"], case["m"], case["n"]
    if f == "uniform":
        return m, n, m * case["longest"] // 2
    if f == "powerlaw":
        return m, n, case["nnz"]
    if f == "laplace":
        s = case["side"]
        return m, n, 7 * m - 6 * s * s
    if f == "banded":
        h = (case["bandwidth"] - 1) // 2
        return m, n, m * case["bandwidth"] - h * (h + 1)
    return m, n, 27 * m


def work(case):
    """A read once, x read once, y written once: per SpMV in a loop; in a batch A
    once, x and y per right-hand side."""
    v = np.dtype(case["dtype"]).itemsize
    if case["kind"] == "batch":
        nbytes = flops = 0
        for m, k, f, p in _batch_sizes(case):
            # a power law's mean row: about 12 entries over its exponents
            nnz = m * (p // 2 if f == "uniform" else 12 if f == "powerlaw" else
                       min(p, m) if f == "banded" else 27)
            nbytes += nnz * (v + 4) + 4 * (m + 1) + 2 * m * k * v
            flops += 2 * nnz * k
        return {"bytes": nbytes, "flops": flops}
    m, n, nnz = _count(case)
    runs = case.get("runs", 1)
    return {"bytes": runs * (nnz * (v + 4) + 4 * (m + 1) + (m + n) * v), "flops": 2.0 * runs * nnz}


def _product(A, X, alpha):
    """alpha A X in 64 bits: products, then a sum over each row's entries."""
    v = A.val.astype(np.float64)
    y = np.zeros((A.m, X.shape[1]))
    rows = np.flatnonzero(np.diff(A.row_ptr))
    for r in range(X.shape[1] if len(rows) else 0):
        x = X[:, r].astype(np.float64)
        y[rows, r] = np.add.reduceat(v * x[A.col], A.row_ptr[rows])
    return alpha * y


def exact(case, seed):
    if case["kind"] == "batch":
        mats, _, Xs = _batch(case, seed)
        return [_product(A, X, case["alpha"]) for A, X in zip(mats, Xs)]
    A, x = _matrix(case, seed)
    return _product(A, x[:, None], case["alpha"])[:, 0]
