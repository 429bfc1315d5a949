"""The one-wave-per-tile kernel against the lane-exact model and the tile loop
(GPU): y must be the same bits for every tile shape it is built for, with the
rows that cross logical waves finished inside the launch, and with the rows
found inside it (the allocation-free entry point)."""
import ctypes as C

import numpy as np
import pytest

import cases
import kernel_model as km
from benchmark_spmv_using_csr_amd import _lib, batched, matgen
from benchmark_spmv_using_csr_amd.spmv import bhsparse_spmv
from test_zz_no_alloc import DeviceArrays, call_noalloc, hip

pytestmark = pytest.mark.gpu


def lengths_around(P, T, waves, seed):
    """Row lengths over `waves` logical waves of T tiles of P nonzeros that meet
    tile and wave ends every way: rows ending on them and one to either side,
    rows inside a tile, over a tile, over two and many logical waves, runs of
    empty rows across the ends; empty rows first and last."""
    rng = np.random.default_rng(seed)
    lens, at = [0] * 7, 0
    total = waves * P * T + 13

    def add(n):
        nonlocal at
        lens.append(int(n))
        at += int(n)

    kind = 0
    while at < total:
        kind += 1
        to_tile, to_wave = P - at % P, P * T - at % (P * T)
        pick = kind % 9
        if pick == 0:
            add(to_tile)                        # ends on a tile's end
        elif pick == 1:
            add(to_wave)                        # ends on a logical wave's end
            lens.extend([0] * int(rng.integers(1, 4)))
        elif pick == 2:
            add(to_wave + 1)
        elif pick == 3:
            add(max(to_wave - 1, 1))
            add(2)                              # one item on each side of the end
        elif pick == 4:
            add(to_wave + P * T)                # the rest of this wave and all of the next
        elif pick == 5 and kind % 2:
            add(to_wave + 2 * P * T + 5)        # four waves
        elif pick == 6:
            lens.extend([0] * int(rng.choice([3, 70, 150, 300])))
            add(3)
        else:
            for n in rng.integers(1, 40, 30):
                add(n)
                if rng.random() < 0.1:
                    lens.append(0)
    return lens + [0] * 5


@pytest.mark.parametrize("S", [4, 8, 16])
@pytest.mark.parametrize("T", [1, 2, 4, 8])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_every_shape_against_the_model(S, T, dtype):
    # over 32 logical waves, so that T > 1 leaves the tile loop too
    c = cases.from_lengths(f"S={S} T={T}", lengths_around(64 * S, T, 40, 10 * S + T),
                           n=4 * 64 * S * T + 100, seed=S)
    c.val = c.val.astype(dtype)
    c.x = c.x.astype(dtype)
    assert c.nnz > 33 * 64 * S * T
    for wpb in (1, 4):
        op = bhsparse_spmv(dtype)
        _lib.check(op.init_platform(0), "init_platform")
        _lib.check(op.set_config(0, S, wpb, T, 0), "set_config")
        y = np.full(c.m, np.nan, dtype)
        _lib.check(op.prepare_mem(c.m, c.n, c.nnz, c.row_ptr, c.col, c.val, c.x, y), "prepare_mem")
        print(f"[gpu] tiles S={S} T={T} wpb={wpb} {np.dtype(dtype).name} nnz={c.nnz}", flush=True)
        ym = km.segsum(c.row_ptr, c.col, c.val, c.x, S=S, TPW=T, alpha=0.75, dtype=dtype)
        for _ in range(2):                      # a second call finds its words empty
            _lib.check(op.spmv(0.75), "spmv")
            _lib.check(op.get_y(), "get_y")
            assert np.array_equal(y, ym), np.flatnonzero(y != ym)[:8]
        op.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_rows_over_many_logical_waves(dtype):
    """Rows over 3, 63, 64, 65 and 200 logical waves (windows of 64 partials),
    between short ones."""
    PW = 64 * 4
    lens = [5, 3 * PW, 9, 63 * PW + 7, 1, 64 * PW, 2, 65 * PW - 3, 0, 4, 200 * PW + 1, 6]
    c = cases.from_lengths("long rows", lens, n=201 * PW, seed=3)
    v, x = c.val.astype(dtype), c.x.astype(dtype)
    op = bhsparse_spmv(dtype)
    _lib.check(op.init_platform(0), "init_platform")
    _lib.check(op.set_config(0, 4, 1, 1, 0), "set_config")
    y = np.zeros(c.m, dtype)
    _lib.check(op.prepare_mem(c.m, c.n, c.nnz, c.row_ptr, c.col, v, x, y), "prepare_mem")
    print(f"[gpu] rows over many waves {np.dtype(dtype).name}", flush=True)
    ym = km.segsum(c.row_ptr, c.col, v, x, S=4, TPW=1, dtype=dtype)
    for _ in range(3):
        _lib.check(op.spmv(1.0), "spmv")
        _lib.check(op.get_y(), "get_y")
        assert np.array_equal(y, ym)


def row_layouts():
    rng = np.random.default_rng(8)
    even = np.full(60_000, 9)
    skewed = np.concatenate([np.full(40_000, 1), np.full(20_000, 25)])
    late = np.concatenate([np.zeros(50_000, int), rng.integers(0, 20, 30_000), np.zeros(40_000, int)])
    pareto = np.minimum((rng.pareto(1.0, 50_000) * 2).astype(int), 30_000)
    holes = np.tile(np.r_[np.full(300, 8), np.zeros(5000, int)], 20)
    mirrored = np.concatenate([np.full(9000, 3), np.full(9000, 15), np.full(9000, 15),
                               np.full(9000, 3)])        # the middle row is where even rows put it
    return {"even": even, "skewed": skewed, "empty ends": late, "pareto": pareto, "holes": holes,
            "mirrored": mirrored, "few rows": np.full(255, 300), "257 rows": np.full(257, 300),
            "one row": np.array([300_000])}


@pytest.mark.parametrize("name", list(row_layouts()))
def test_rows_found_inside_the_launch(name):
    """Against a handle with the default tile, whose rows partition_kernel finds."""
    lens = row_layouts()[name]
    rng = np.random.default_rng(len(lens))
    m, n, nnz = len(lens), 300_000, int(lens.sum())
    row_ptr = np.r_[0, np.cumsum(lens)].astype(np.int32)
    col = rng.integers(0, n, nnz).astype(np.int32)
    val, x = rng.uniform(-1, 1, nnz), rng.uniform(-1, 1, n)
    print(f"[gpu] rows found inside the launch: {name} m={m} nnz={nnz}", flush=True)
    op = bhsparse_spmv(np.float64)
    _lib.check(op.init_platform(0), "init_platform")
    y = np.zeros(m)
    _lib.check(op.prepare_mem(m, n, nnz, row_ptr, col, val, x, y), "prepare_mem")
    _lib.check(op.spmv(-0.5), "spmv")
    _lib.check(op.get_y(), "get_y")
    with DeviceArrays(row_ptr, col, val, x, np.full(m, np.nan)) as d:
        for _ in range(2):
            _lib.check(call_noalloc(np.float64, m, n, nnz, d.ptrs, -0.5), "spmv_noalloc")
            assert np.array_equal(d.get(4, y), y)


def test_beyond_the_one_kernel_sizes():
    """More logical waves than the one-kernel path has words for (134M nonzeros):
    partition, kernel and calibration; whole numbers, so the sums are exact."""
    nnz, m, n = 65536 * 2048 + 3001, 1_000_003, 1000
    row_ptr = (np.arange(m + 1, dtype=np.int64) * nnz // m).astype(np.int32)
    row_ptr[500_001:500_020] = row_ptr[500_020]                   # a row of 2,700 and empty rows
    col = np.arange(nnz, dtype=np.int32) % n
    x = (np.arange(n) % 7 - 3).astype(np.float32)
    print(f"[gpu] {nnz} nonzeros through spmv_noalloc", flush=True)
    sums = np.r_[0, np.cumsum(x.astype(np.int64)[col])]
    y0 = np.full(m, np.nan, np.float32)
    with DeviceArrays(row_ptr, col, np.ones(nnz, np.float32), x, y0) as d:
        _lib.check(call_noalloc(np.float32, m, n, nnz, d.ptrs, 1.0), "spmv_noalloc")
        y = d.get(4, y0)
    assert np.array_equal(y.astype(np.int64), sums[row_ptr[1:]] - sums[row_ptr[:-1]])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_more_logical_waves_than_the_fused_launch_takes(dtype):
    """A handle's default tile over 16,384 logical waves (kernel, then
    calibration) against the allocation-free entry point (one kernel)."""
    A = matgen.uniform_rows(21, 1_300_000, 900_000, 0, 56)
    assert A.nnz > 16384 * 2048
    v, x = A.val.astype(dtype), matgen.vector(22, A.n).astype(dtype)
    print(f"[gpu] {A.nnz} nonzeros {np.dtype(dtype).name}", flush=True)
    op = bhsparse_spmv(dtype)
    _lib.check(op.init_platform(0), "init_platform")
    y = np.zeros(A.m, dtype)
    _lib.check(op.prepare_mem(A.m, A.n, A.nnz, A.row_ptr, A.col, v, x, y), "prepare_mem")
    _lib.check(op.spmv(1.5), "spmv")
    _lib.check(op.get_y(), "get_y")
    with DeviceArrays(A.row_ptr, A.col, v, x, np.full(A.m, np.nan, dtype)) as d:
        _lib.check(call_noalloc(dtype, A.m, A.n, A.nnz, d.ptrs, 1.5), "spmv_noalloc")
        assert np.array_equal(d.get(4, y), y)


@pytest.mark.parametrize("S", [4, 8, 16])
@pytest.mark.parametrize("T", [1, 2, 4, 8])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_batches_against_the_tile_loop(S, T, dtype):
    """Even and odd numbers of right-hand sides over matrices whose rows meet tile
    and wave ends every way, and the shapes with nothing to do, against one plain
    SpMV (the tile loop) per matrix and right-hand side."""
    cs = [cases.from_lengths(f"around {i}", lengths_around(64 * S, T, 6, 100 * S + 10 * T + i),
                             n=4 * 64 * S * T + 100, seed=i) for i in range(4)]
    cs += [cases.from_lengths("empty", [0] * 9, seed=1), cases.six_by_six(),
           cases.from_lengths("lead", [0] * 3000 + [2] * 5, seed=2),
           cases.from_lengths("one row", [5 * 64 * S * T + 3], seed=3)]
    mats = [matgen.CSR(c.m, c.n, c.row_ptr, c.col, c.val.astype(dtype), c.name) for c in cs]
    ks = [1, 2, 3, 16, 4, 5, 2, 16]
    rng = np.random.default_rng(S * T)
    Xs = [rng.uniform(-1, 1, (A.n, k)).astype(dtype) for A, k in zip(mats, ks)]
    print(f"[gpu] batch S={S} T={T} {np.dtype(dtype).name}", flush=True)
    b = batched.SpmvBatch(mats, ks, dtype)
    b.set_schedule(S, T, 1, 0, 1, 0)
    for turn in range(2):                       # the second run overwrites the first one's y
        b.set_x([X * (turn + 1) for X in Xs])
        b.run(0.75)
        b.run_plain(0.75)
        for i, (yb, yp) in enumerate(zip(b.y(), b.y(plain=True))):
            assert np.array_equal(yb, yp), (i, mats[i].name, ks[i])
    b.close()


def leading(lead, P, tiles, seed):
    """`lead` empty rows, then rows with entries over `tiles` tiles of P."""
    rng = np.random.default_rng(seed)
    lens = [0] * lead
    while sum(lens) < tiles * P - 30:
        lens.append(int(rng.integers(1, 30)))
    return lens


# fewer empty rows than tiles, than lanes, and about their multiples: some waves
# have no share of them, some a part of one
LEADS = [1, 2, 63, 64, 65, 129, 1000, 4097]


@pytest.mark.parametrize("tiles", [1, 3, 50, 131])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_leading_empty_rows_and_the_rows_behind_them(tiles, dtype):
    """The leading empty rows are zeroed by shares and the rows behind them keep
    their sums: on a handle, with the rows found inside the launch, and in a batch."""
    cs = [cases.from_lengths(f"lead {lead}", leading(lead, 512, tiles, lead), n=5000, seed=lead)
          for lead in LEADS]
    print(f"[gpu] leading empty rows, {tiles} tiles, {np.dtype(dtype).name}", flush=True)
    want = [km.segsum(c.row_ptr, c.col, c.val.astype(dtype), c.x.astype(dtype), S=8, TPW=1,
                      alpha=0.5, dtype=dtype) for c in cs]
    four = [km.segsum(c.row_ptr, c.col, c.val.astype(dtype), c.x.astype(dtype), S=8, TPW=4,
                      alpha=0.5, dtype=dtype) for c in cs]
    for c, w1, w4 in zip(cs, want, four):
        v, x = c.val.astype(dtype), c.x.astype(dtype)
        op, y = bhsparse_spmv(dtype), np.full(c.m, np.nan, dtype)
        _lib.check(op.init_platform(0), "init_platform")
        _lib.check(op.set_config(0, 8, 4, 1, 0), "set_config")
        _lib.check(op.prepare_mem(c.m, c.n, c.nnz, c.row_ptr, c.col, v, x, y), "prepare_mem")
        _lib.check(op.spmv(0.5), "spmv")
        _lib.check(op.get_y(), "get_y")
        op.close()
        assert np.array_equal(y, w1), c.name
        with DeviceArrays(np.asarray(c.row_ptr, np.int32), np.asarray(c.col, np.int32), v, x,
                          np.full(c.m, np.nan, dtype)) as d:
            _lib.check(call_noalloc(dtype, c.m, c.n, c.nnz, d.ptrs, 0.5), "spmv_noalloc")
            assert np.array_equal(d.get(4, y), w4), c.name
    mats = [matgen.CSR(c.m, c.n, c.row_ptr, c.col, c.val.astype(dtype), c.name) for c in cs]
    ks = [(1, 2, 3, 16)[i % 4] for i in range(len(cs))]
    b = batched.SpmvBatch(mats, ks, dtype)
    b.set_x([np.repeat(c.x.astype(dtype)[:, None], k, 1) for c, k in zip(cs, ks)])
    b.set_schedule(8, 1, 1, 0, 1, 0)
    b.run(0.5)
    for Y, w1, c in zip(b.y(), want, cs):
        assert np.array_equal(Y, np.repeat(w1[:, None], Y.shape[1], 1)), c.name
    b.close()


@pytest.mark.parametrize("empty", [(1 << 30) + 7, 1_500_000_001])
def test_more_empty_rows_than_half_the_index_range(empty):
    """A run of over 2^30 empty rows between two groups of rows with entries: the
    steps along it do not pass 2^31.  Whole numbers; y is read at both ends of the
    run and at places inside."""
    H = hip()
    H.hipMemsetD32.argtypes = [C.c_void_p, C.c_int, C.c_size_t]
    lens = [3] * 900
    rp = np.cumsum([0] + lens).astype(np.int32)
    m, half = empty + 1800, int(rp[-1])
    nnz, n = 2 * half, 1000
    rng = np.random.default_rng(1)
    col = rng.integers(0, n, nnz).astype(np.int32)
    val = rng.integers(-3, 4, nnz).astype(np.float32)
    x = rng.integers(-3, 4, n).astype(np.float32)
    want = np.add.reduceat(val * x[col], np.arange(0, nnz, 3))
    ptr = {}
    try:
        for name, words in (("row_ptr", m + 1), ("y", m)):
            ptr[name] = C.c_void_p()
            assert H.hipMalloc(C.byref(ptr[name]), 4 * words) == 0
        at = lambda name, i: C.c_void_p(ptr[name].value + 4 * i)
        assert H.hipMemsetD32(ptr["row_ptr"], half, m + 1) == 0
        assert H.hipMemsetD32(ptr["y"], 0x7fc00000, m) == 0            # NaN
        assert H.hipMemcpy(at("row_ptr", 0), rp.ctypes.data_as(C.c_void_p), rp.nbytes, 1) == 0
        tail = rp + np.int32(half)
        assert H.hipMemcpy(at("row_ptr", m - 900), tail.ctypes.data_as(C.c_void_p), tail.nbytes,
                           1) == 0
        print(f"[gpu] {empty} empty rows in a row", flush=True)
        with DeviceArrays(col, val, x) as d:
            _lib.check(call_noalloc(np.float32, m, n, nnz,
                                    [ptr["row_ptr"], *d.ptrs, ptr["y"]], 1.0), "spmv_noalloc")
            assert H.hipDeviceSynchronize() == 0
        def y(lo, hi):
            out = np.empty(hi - lo, np.float32)
            assert H.hipMemcpy(out.ctypes.data_as(C.c_void_p), at("y", lo), out.nbytes, 2) == 0
            return out
        assert np.array_equal(y(0, 900), want[:900])
        assert np.array_equal(y(m - 900, m), want[900:])
        for lo in (900, 5000, 1 << 29, 1 << 30, m // 2, m - 900 - 70_000):
            assert not y(lo, min(lo + 70_000, m - 900)).any()
    finally:
        for p in ptr.values():
            H.hipFree(p)


@pytest.mark.parametrize("T", [1, 4])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_long_rows_counted_by_groups(T, dtype):
    """Rows over 63 to 300 logical waves whose first and last waves lie on, before
    and behind the ends of groups of 32, one behind the other (the last wave of
    one is the first of the next) and with short ones between."""
    PW, lens, at = 64 * 4 * T, [], 0

    def to(wave, inside):                      # a row up to `inside` nonzeros into a wave
        nonlocal at
        lens.append(wave * PW + inside - at)
        at = wave * PW + inside

    for wave, inside in [(0, 5), (63, 9), (64, 3), (127, 7), (128, 1), (193, 2), (256, 4), (321, PW),
                         (352, 11), (417, 8), (482, 6), (546, PW), (578, 1), (578, 40), (672, 1),
                         (735, 5), (736, 5), (1036, 9)]:
        to(wave, inside)
    lens += [3, 0, 2]
    c = cases.from_lengths("groups", lens, n=5000, seed=T)
    v, x = c.val.astype(dtype), c.x.astype(dtype)
    op, y = bhsparse_spmv(dtype), np.zeros(c.m, dtype)
    _lib.check(op.init_platform(0), "init_platform")
    _lib.check(op.set_config(0, 4, 1, T, 0), "set_config")
    _lib.check(op.prepare_mem(c.m, c.n, c.nnz, c.row_ptr, c.col, v, x, y), "prepare_mem")
    print(f"[gpu] long rows by groups T={T} {np.dtype(dtype).name} nnz={c.nnz}", flush=True)
    ym = km.segsum(c.row_ptr, c.col, v, x, S=4, TPW=T, dtype=dtype)
    for _ in range(3):
        _lib.check(op.spmv(1.0), "spmv")
        _lib.check(op.get_y(), "get_y")
        assert np.array_equal(y, ym), np.flatnonzero(y != ym)
    op.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_long_rows_found_inside_the_launch(dtype):
    """Rows over 70 to 2,500 logical waves of the default tile through the
    allocation-free entry point; whole numbers."""
    lens = [4, 70 * 2048 + 3, 0, 9, 700 * 2048, 1, 2500 * 2048 + 77, 5]
    row_ptr = np.r_[0, np.cumsum(lens)].astype(np.int32)
    m, n, nnz = len(lens), 1000, int(row_ptr[-1])
    col = np.arange(nnz, dtype=np.int32) % n
    x = (np.arange(n) % 7 - 3).astype(dtype)
    val = np.ones(nnz, dtype)
    print(f"[gpu] {nnz} nonzeros in {m} rows {np.dtype(dtype).name}", flush=True)
    sums = np.r_[0, np.cumsum(x.astype(np.int64)[col])]
    y0 = np.full(m, np.nan, dtype)
    with DeviceArrays(row_ptr, col, val, x, y0) as d:
        for _ in range(2):
            _lib.check(call_noalloc(dtype, m, n, nnz, d.ptrs, 2.0), "spmv_noalloc")
            y = d.get(4, y0)
            assert np.array_equal(y.astype(np.int64), 2 * (sums[row_ptr[1:]] - sums[row_ptr[:-1]]))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_runs_of_empty_rows_at_every_alignment(dtype):
    """Runs of 128 to 1,500 empty rows that start and end at every offset from 16
    bytes, y itself at each of them; the values before and behind y stay."""
    rng = np.random.default_rng(5)
    lens = []
    for run in [128, 129, 130, 131, 255, 256, 257, 700, 1001, 1002, 1003, 1500]:
        lens += list(rng.integers(1, 4, int(rng.integers(1, 6)))) + [0] * run
    lens += [2, 1]
    c = cases.from_lengths("runs", lens, n=3000, seed=6)
    v, x = c.val.astype(dtype), c.x.astype(dtype)
    want = km.segsum(c.row_ptr, c.col, v, x, S=8, TPW=4, dtype=dtype)
    print(f"[gpu] runs of empty rows {np.dtype(dtype).name}", flush=True)
    room = np.full(c.m + 16, 7, dtype)
    for off in range(16 // room.itemsize):
        with DeviceArrays(np.asarray(c.row_ptr, np.int32), np.asarray(c.col, np.int32), v, x,
                          room) as d:
            y = C.c_void_p(d.ptrs[4].value + (4 + off) * room.itemsize)
            _lib.check(call_noalloc(dtype, c.m, c.n, c.nnz, [*d.ptrs[:4], y], 1.0), "spmv_noalloc")
            got = d.get(4, room)
        assert np.array_equal(got[4 + off:4 + off + c.m], want), off
        assert np.all(got[:4 + off] == 7) and np.all(got[4 + off + c.m:] == 7)
    for tile in [(0, 8, 4, 1, 0), (0, 4, 1, 16, 0)]:          # a wave per tile; the tile loop
        op, y = bhsparse_spmv(dtype), np.full(c.m, np.nan, dtype)
        _lib.check(op.init_platform(0), "init_platform")
        _lib.check(op.set_config(*tile), "set_config")
        _lib.check(op.prepare_mem(c.m, c.n, c.nnz, c.row_ptr, c.col, v, x, y), "prepare_mem")
        _lib.check(op.spmv(1.0), "spmv")
        _lib.check(op.get_y(), "get_y")
        op.close()
        assert np.array_equal(y, km.segsum(c.row_ptr, c.col, v, x, S=tile[1], TPW=tile[3],
                                           dtype=dtype)), tile
    A = matgen.CSR(c.m, c.n, c.row_ptr, c.col, v, c.name)
    for T in (4, 16):                                         # a wave per tile; the tile loop
        b = batched.SpmvBatch([A] * 4, [1, 2, 3, 16], dtype)
        b.set_schedule(8, T, 1, 0, 1, 0)
        b.set_x([np.repeat(x[:, None], k, 1) for k in (1, 2, 3, 16)])
        b.run(1.0)
        b.run_plain(1.0)
        for Y, P in zip(b.y(), b.y(plain=True)):
            assert np.array_equal(Y, P) and not np.isnan(Y).any()
        b.close()


def rows_over_waves(PW, waves, lead, seed):
    """Rows over 3, 64, 65 and 200 logical waves, rows that end on a wave's end and
    one to either side, runs of empty rows at wave ends and inside, `lead` empty rows
    first; the mean row is longer than a logical wave."""
    rng = np.random.default_rng(seed)
    lens, at = [0] * lead, 0

    def to(n):
        nonlocal at
        lens.append(n)
        at += n

    long = [3 * PW + 7, 64 * PW, 65 * PW - 5, 200 * PW + 1, 2 * PW]
    while at < waves * PW:
        left = PW - at % PW
        pick = rng.integers(0, 7)
        if pick == 0 and long:
            to(long.pop())
        elif pick == 1:
            to(left)
            lens += [0] * int(rng.integers(0, 4))
        elif pick == 2:
            to(left + PW)
            lens += [0] * int(rng.choice([0, 70, 140]) if len(lens) < 300 else 0)
        elif pick == 3:
            to(left + 1)
        elif pick == 4:
            to(left + 2 * PW - 1)
            to(2)
        else:
            to(left + int(rng.integers(1, 4 * PW)))
    for n in long:
        to(n)
    return lens + [0] * 3


@pytest.mark.parametrize("S,T", [(4, 2), (4, 8), (8, 2), (8, 4), (16, 2), (16, 4)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_rows_left_to_the_calibration(S, T, dtype):
    """One wave per tile without the fused end: rows that pass through whole logical
    waves, and leading empty rows.  Whole numbers, so the sums are exact."""
    from test_gpu_choice import kernels_of_a_call
    for lead in (0, 1, 65, 500):
        lens = rows_over_waves(64 * S * T, 1300, lead, 10 * S + T + lead)
        row_ptr = np.r_[0, np.cumsum(lens)].astype(np.int32)
        m, n, nnz = len(lens), 3000, int(row_ptr[-1])
        assert nnz > 64 * S * T * m
        rng = np.random.default_rng(S + T)
        col = rng.integers(0, n, nnz).astype(np.int32)
        val, x = rng.integers(-3, 4, nnz), rng.integers(-3, 4, n)
        sums = np.r_[0, np.cumsum(val * x[col])]
        op, y = bhsparse_spmv(dtype), np.full(m, np.nan, dtype)
        _lib.check(op.init_platform(0), "init_platform")
        _lib.check(op.set_config(0, S, 4, T, 0), "set_config")
        _lib.check(op.prepare_mem(m, n, nnz, row_ptr, col, val.astype(dtype), x.astype(dtype), y),
                   "prepare_mem")
        print(f"[gpu] left to the calibration: S={S} T={T} lead={lead} nnz={nnz} "
              f"{np.dtype(dtype).name}", flush=True)
        assert kernels_of_a_call(op) == 2
        for alpha in (1.0, -2.0):
            _lib.check(op.spmv(alpha), "spmv")
            _lib.check(op.get_y(), "get_y")
            assert np.array_equal(y, alpha * (sums[row_ptr[1:]] - sums[row_ptr[:-1]]))
        op.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_rows_left_to_the_calibration_bit_for_bit(dtype):
    """The same kind of rows at the default tile against the allocation-free entry
    point, whose launch finishes them itself."""
    from test_gpu_choice import kernels_of_a_call
    lens = rows_over_waves(2048, 1300, 65, 1)
    row_ptr = np.r_[0, np.cumsum(lens)].astype(np.int32)
    m, n, nnz = len(lens), 40_000, int(row_ptr[-1])
    rng = np.random.default_rng(2)
    col = rng.integers(0, n, nnz).astype(np.int32)
    val, x = rng.uniform(-1, 1, nnz).astype(dtype), rng.uniform(-1, 1, n).astype(dtype)
    op, y = bhsparse_spmv(dtype), np.full(m, np.nan, dtype)
    _lib.check(op.init_platform(0), "init_platform")
    _lib.check(op.prepare_mem(m, n, nnz, row_ptr, col, val, x, y), "prepare_mem")
    assert kernels_of_a_call(op) == 2
    _lib.check(op.spmv(0.75), "spmv")
    _lib.check(op.get_y(), "get_y")
    op.close()
    with DeviceArrays(row_ptr, col, val, x, np.full(m, np.nan, dtype)) as d:
        _lib.check(call_noalloc(dtype, m, n, nnz, d.ptrs, 0.75), "spmv_noalloc")
        assert np.array_equal(d.get(4, y), y)
