// bhs_kernels.h -- gfx950 kernels of the speculative segmented-sum SpMV.
//
// Data layout in HBM (all 0-based CSR, 32-bit indices):
//   row_ptr  (m+1) int          col  nnz_pad int (nontemporal stream)
//   val      nnz_pad T (stream)  x    n T (gathered, cached)    y  m T
//   tile_row NP+1 int  -- first row of every tile boundary, computed once
//   sync_row / sync_val  NW entries -- boundary-row partial of every wave
// nnz_pad rounds nnz up to whole tiles of the largest shape, padded with
// col = 0 / val = 0, so every lane loads its items without bounds checks.
//
// A tile is P = 64*S consecutive nonzeros (S items per lane); a wave walks
// TPW consecutive tiles carrying the open row's partial sum from tile to tile,
// as a thread bunch walks STEP tiles in the reference (spmv_cuda/common.h:39-48,
// kernels_cuda.h:64).
#pragma once
#include "bhs_device.h"

namespace bhs {

// ---------------------------------------------------------------------------
// Partition: tile_row[p] = upper_bound(row_ptr[0..m], min(p*P, nnz)) - 1.
// Same bisection as binary_search_right_boundary_kernel (utils_cuda.h:6-34)
// applied to every tile boundary (kernels_cuda.h:43-49); it depends only on
// row_ptr and P, so it runs once per matrix and tile size, not per call.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void partition_kernel(const int *__restrict__ row_ptr, int m,
                                                       int nnz, int P, int NP,
                                                       int *__restrict__ tile_row)
{
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p > NP) return;
    long long k = p * (long long)P;
    const int key = k > nnz ? nnz : (int)k;
    int lo = 0, hi = m + 1;                  // search [lo, hi) of row_ptr[0..m]
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (row_ptr[mid] <= key) lo = mid + 1;
        else hi = mid;
    }
    tile_row[p] = lo - 1;
}

// Scalars of one launch (the arrays travel as separate __restrict__ kernel
// arguments, which lets the compiler use scalar loads for tile_row/row_ptr).
template <typename T>
struct SegsumParams {
    int m, nnz, NP, TPW, NW, lead_empty, wpb, wave_lds_bytes;
    T alpha;
    long long x_lines;   // > 0: x is read ahead into each XCD's L2 (x_lines 128-byte lines)
    int x_far;           // x reaches past 4 GB (64-bit gather addresses)
};

// One tile's column indices and values in registers.  Loads are coalesced:
// for load group j, lane l reads G = 16/sizeof(T) consecutive items starting at
// B + j*64*G + l*G (consecutive lanes read consecutive 16-byte values), so item
// k = j*G + g of lane l is nonzero B + j*64*G + l*G + g.
template <typename T, int S>
struct Tile {
    static constexpr int G = 16 / (int)sizeof(T);
    static constexpr int J = S / G;
    static_assert(S % G == 0 && S >= 4, "S must be a multiple of 16 / sizeof(T) and >= 4");
    int c[S];
    T v[S];
};

template <typename T, int S>
__device__ __forceinline__ int tile_item(int B, int lane, int k)
{
    constexpr int G = Tile<T, S>::G;
    return B + (k / G) * (kWave * G) + lane * G + (k % G);
}

template <typename T, int S>
__device__ __forceinline__ void tile_load(const int *__restrict__ col, const T *__restrict__ val,
                                          int B, int lane, Tile<T, S> &t)
{
    constexpr int G = Tile<T, S>::G, J = Tile<T, S>::J;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int e = B + j * (kWave * G) + lane * G;
        const u32x4 qv = load_nt16(val + e);
        __builtin_memcpy(&t.v[j * G], &qv, 16);
        if constexpr (G == 4) {
            const u32x4 qc = load_nt16(col + e);
            t.c[j * 4 + 0] = (int)qc.x;
            t.c[j * 4 + 1] = (int)qc.y;
            t.c[j * 4 + 2] = (int)qc.z;
            t.c[j * 4 + 3] = (int)qc.w;
        } else {
            const u32x2 qc = load_nt8(col + e);
            t.c[j * 2 + 0] = (int)qc.x;
            t.c[j * 2 + 1] = (int)qc.y;
        }
    }
}

// The same items with every index checked against nnz (items past it read
// as col 0 / val 0): the last tile of a matrix whose arrays are not padded.
template <typename T, int S>
__device__ __forceinline__ void tile_load_checked(const int *__restrict__ col,
                                                  const T *__restrict__ val, int B, int lane,
                                                  int nnz, Tile<T, S> &t)
{
#pragma unroll
    for (int k = 0; k < S; ++k) {
        const int e = tile_item<T, S>(B, lane, k);
        t.c[k] = e < nnz ? col[e] : 0;
        t.v[k] = e < nnz ? val[e] : T(0);
    }
}

// Row boundaries of the first 64*CP rows of a tile starting at row r (CP = 2
// or 4 chunk parts): lane l holds a[q] = row_ptr[r + 64q + l] for q < CP, and
// every lane holds end = row_ptr[r + 64*CP], each index clamped to m (row_ptr
// has m+1 entries, so every address is in bounds; callers ignore rows past the
// tile's last row).  A row's end, row_ptr[r + 64q + l + 1], is lane l+1's a[q]
// (lane 63: a[q+1] of lane 0, or end), so CP loads per lane cover 64*CP rows.
// Loaded one tile ahead of its use.  CP = 4 pays on matrices where many tiles
// span 128-255 rows (short rows), CP = 2 elsewhere; the host picks per matrix.
template <int CP>
struct RowChunk {
    int a[CP];
    int end;
};

template <int CP>
__device__ __forceinline__ RowChunk<CP> load_chunk(const int *__restrict__ row_ptr, int r,
                                                   int lane, int m)
{
    RowChunk<CP> c;
    static_for<CP>([&](auto qc) { c.a[qc] = row_ptr[min(r + qc * kWave + lane, m)]; });
    c.end = row_ptr[min(r + CP * kWave, m)];
    return c;
}

// row_ptr[r + 64Q + lane + 1] from a chunk loaded at row r.  Reads other
// lanes: call it with every lane of the wave active.
template <int Q, int CP>
__device__ __forceinline__ int chunk_next(const RowChunk<CP> &c, int lane)
{
    int first_after;
    if constexpr (Q + 1 < CP) first_after = read_lane(c.a[Q + 1], 0);
    else first_after = c.end;
    const int up = dpp<kDppWaveShl1>(c.a[Q], first_after);
    return lane == kWave - 1 ? first_after : up;
}

// Number of tiles p < NP whose row span tile_row[p+1] - tile_row[p] lies in
// [lo, hi), added to *count (one atomic per wave).
__global__ __launch_bounds__(256) void tile_span_count_kernel(const int *__restrict__ tile_row,
                                                              int NP, int lo, int hi,
                                                              unsigned long long *count)
{
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    bool in = false;
    if (p < NP) {
        const int d = tile_row[p + 1] - tile_row[p];
        in = d >= lo && d < hi;
    }
    const uint64_t b = ballot(in);
    if (lane_id() == 0 && b) atomicAdd(count, (unsigned long long)__popcll(b));
}

// Compile-time switch between the tile code paths of segsum_wave.
template <bool B>
struct BigTag {
    static constexpr bool value = B;
};

// Given row_ptr[lo] == v (rows before lo, back to the run's start, are empty),
// the end (exclusive, at most stop+1) of the run of empty rows: the first row
// at or after lo with entries.  Wave-uniform doubling steps over row_ptr,
// closed by bisection, so a tile spanning a long run of empty rows costs
// O(log run) loads instead of one per row.
__device__ __forceinline__ int empty_run_end(const int *__restrict__ row_ptr, int lo, int v,
                                             int stop)
{
    unsigned step = 64;                      // steps by their length: lo + step may pass 2^31
    while (step <= (unsigned)(stop + 1 - lo) && row_ptr[lo + step] == v) {
        lo += step;
        step *= 2;
    }
    int hi = lo + (int)min(step, (unsigned)(stop + 1 - lo));
    if (row_ptr[hi] == v) return stop + 1;   // empty up to the tile's last row
    while (hi - lo > 1) {                    // row_ptr[lo] == v < row_ptr[hi]
        const int mid = lo + (hi - lo) / 2;
        if (row_ptr[mid] == v) lo = mid;
        else hi = mid;
    }
    return lo;
}

// y[lo, hi) = 0 by one wave, 16 bytes a lane: a wave has 63 stores on their way at
// most, so a long run's time is their number (300,000 rows at the end of a matrix of
// 450,000 nonzeros, a call, fp64 / fp32: 150 / 149 us with a value a lane, 69 / 38).
template <typename T>
__device__ __forceinline__ void zero_run(T *__restrict__ y, long long lo, long long hi, int lane)
{
    constexpr int N = 16 / (int)sizeof(T);
    const int head = (int)(-(reinterpret_cast<uintptr_t>(y + lo) / sizeof(T)) & (N - 1));
    if (lane < head && lo + lane < hi) y[lo + lane] = T(0);
    long long r = lo + head + lane * N;
    for (; r + N <= hi; r += kWave * N)
        *reinterpret_cast<u32x4 *>(y + r) = u32x4{0u, 0u, 0u, 0u};
    for (; r < hi; ++r) y[r] = T(0);     // fewer than N rows, in one lane
}

// ---------------------------------------------------------------------------
// Speculative segmented sum (kernels_cuda.h:7-269, wave64 form).
//
// Per tile [B, B+P) with r0 = tile_row[p], r1 = tile_row[p+1]:
//  * products val*x[col] (kernels_cuda.h:150-162): coalesced loads, the x
//    gathers all issued before any of them is waited on; the next tile's
//    col/val stream and the row_ptr values of its first 256 rows are in
//    flight while this tile is reduced, so no tile waits on a row_ptr load
//    unless it spans more than 256 rows.
//  * fast track (r0 == r1, the tile lies inside one row, :79-112): lane sums,
//    wave sum, added to the carried partial; nothing is stored until the row
//    closes.
//  * otherwise
//    - bit flags (:114-148): each lane takes rows r0+l and r0+64+l (further
//      rows, rare, in a loop) of [r0, min(r1, m-1)]; a nonempty
//      row starting at offset o in [0, P) sets bit o%S of lane o/S's word
//      (LDS atomic OR); an empty row marks the tile dirty and gets y = 0.
//    - the products go through LDS so lane l owns items [lS, lS+S) in order
//      (the reference's s_interres transpose, :150-162).
//    - carry-in (:164-172): if item 0 does not start a row it gets the
//      carried partial added; lane 0's item 0 always starts a segment.
//    - lane-sequential segmented reduction over the S items (:174-203);
//      segments that close inside a lane go straight to LDS s_seg[k].
//    - segment numbers: exclusive wave scan of per-lane head counts (:205-207).
//    - segments spanning lanes (:209-235): a segmented wave scan of the lane
//      tails replaces the reference's O(W) serial walk; the next lane with a
//      head (or lane 63 for the tile's last segment) closes the segment.
//    - speculation: segment k is row r0+k when the tile has no empty row; in
//      a dirty tile the fix-up of bhsparse_spmv_cuda.h:178-222 is done in the
//      wave: rows get their segment by rank among nonempty rows (ballot +
//      mbcnt), so no second pass over y and no host round trip.
//  * The first row of a wave, if it began in an earlier wave, is not stored:
//    its partial goes to sync_val[w] (the reference's synchronizer,
//    :98-102/:243-247) and calibrate_kernel adds it.  The wave in which a row
//    begins stores that row's partial with a plain store, so every call
//    overwrites y completely (beta = 0, repeatable), unlike the reference's
//    y[idx] += of stale values (bhsparse_spmv_cuda.h:170-173).
// ---------------------------------------------------------------------------
// One matrix as one wave sees it.  X is n x kstride and Y is m x kstride,
// row-major (a column's right-hand sides share cache lines); the wave computes
// k of them (k <= KMAX).  Rows' partials that cross waves go to
// sync_row[w] = key_base + row * kstride (the y slot of RHS 0 of the row) and
// sync_val[w * KMAX + rr].
template <typename T>
struct MatView {
    const int *row_ptr;
    const int *tile_row;
    const int *col;
    const T *val;
    const T *x;
    T *y;
    int *sync_row;
    T *sync_val;
    int m, nnz, NP, NW, lead_empty, k, kstride, TPW, key_base;
};

// x values of the tile's items for the right-hand side being reduced (v).
// One right-hand side: a gather per item.  Several (KMAX > 1): the gathers
// of the next right-hand side are issued before the current one is reduced,
// so their latency overlaps that work.
template <typename T, int S, int KMAX>
struct RhsX {
    T v[S];                                     // RHS rr
    T n0[S];                                    // KMAX > 1: RHS rr+1

    __device__ __forceinline__ void load1(const T *__restrict__ x, const Tile<T, S> &t, int ks,
                                          int rr, T (&d)[S])
    {
#pragma unroll
        for (int kk = 0; kk < S; ++kk) d[kk] = x[(long long)t.c[kk] * ks + rr];
    }
    __device__ __forceinline__ void first(const T *__restrict__ x, const Tile<T, S> &t, int ks)
    {
        load1(x, t, ks, 0, v);
    }
    // at the top of RHS rr: the loads of RHS rr+1
    __device__ __forceinline__ void issue(const T *__restrict__ x, const Tile<T, S> &t, int ks,
                                          int rr, int k)
    {
        if constexpr (KMAX > 1)
            if (rr + 1 < k) load1(x, t, ks, rr + 1, n0);
    }
    // at the end of RHS rr: v becomes RHS rr+1
    __device__ __forceinline__ void advance(int rr, int k)
    {
        if constexpr (KMAX > 1) {
            if (rr + 1 >= k) return;
#pragma unroll
            for (int kk = 0; kk < S; ++kk) v[kk] = n0[kk];
        }
    }
};

// Right-hand sides in pairs (k even, even stride, x offsets even): RHS rr and
// rr+1 of an item come from one aligned 2-wide load and are reduced together
// as 2-vectors, each component with exactly the single-RHS arithmetic; the
// next pair's loads are in flight while the current pair is reduced.
template <typename T, int S>
struct RhsPair {
    using V = typename RhsVec<T, 2>::type;
    V v[S], n[S];

    __device__ __forceinline__ void load(const T *__restrict__ x, const Tile<T, S> &t, int ks,
                                         int rr, V (&d)[S])
    {
#pragma unroll
        for (int kk = 0; kk < S; ++kk)
            d[kk] = *reinterpret_cast<const V *>(x + (long long)t.c[kk] * ks + rr);
    }
    __device__ __forceinline__ void first(const T *__restrict__ x, const Tile<T, S> &t, int ks)
    {
        load(x, t, ks, 0, v);
    }
    __device__ __forceinline__ void issue(const T *__restrict__ x, const Tile<T, S> &t, int ks,
                                          int rr, int k)
    {
        if (rr + 2 < k) load(x, t, ks, rr + 2, n);
    }
    __device__ __forceinline__ void advance(int rr, int k)
    {
        if (rr + 2 >= k) return;
#pragma unroll
        for (int kk = 0; kk < S; ++kk) v[kk] = n[kk];
    }
};

// Right-hand sides in pairs with the tile's x values staged in LDS (fp64,
// S = 4, k even): an item's k values are k*8 contiguous bytes of X (one
// 128-byte line at k = 16), cut into C = k/2 16-byte chunks, one pair each.
// Staged XCH chunks at a time (a pass), the chunks of an item come from one
// load instruction, on neighbouring lanes, so each line is one request to
// the cache per pass instead of one per pair; the pairs are then read from
// LDS.  (Loading the next pass into a second buffer while the current one is
// reduced measured slower: the extra LDS costs more resident waves than the
// overlap gains.)
//
// Layout of a pass (Cp = min(C, XCH) rounded up to a power of two, the same
// for every pass of a tile; M = 16/Cp): load instruction i in [0, 4*Cp)
// writes LDS bytes [1024 i, 1024 i + 1024), lane l at 16 l.  Lane l of
// instruction i loads chunk c of item t where, with s = l / Cp, q = l % Cp,
// r = s % M, w = s / M, e = 4 i + w, v = e / 2:
//     t = 2 (v M + r) + e % 2,    c = (q - v) mod Cp.
// A pair read has lane L take item t = 128 j + 2 L + g (fixed j, g) at one
// chunk c: lanes L = 0..15 then land in the 16 distinct 16-byte bank groups
// (r = L mod M, q = (c + L / M) mod Cp), so the reads are conflict-free.
template <int XCH>
struct XStage {
    unsigned char *buf;                            // 1024 * 4 * XCH bytes
    int *s_col;                                    // the tile's column indices
    int lc = 0, lm = 4, q = 0, w = 0, tb = 0;     // the tile's pass geometry, this lane

    // The tile's columns (lane L holds items 128j+2L+g) and the pass geometry:
    // the item this lane loads in instruction i is tb + i * 4M.
    __device__ __forceinline__ void begin_tile(const Tile<double, 4> &t, int lane, int C)
    {
        wave_sync();                               // earlier reads of s_col are done
        s_col[2 * lane] = t.c[0];
        s_col[2 * lane + 1] = t.c[1];
        s_col[128 + 2 * lane] = t.c[2];
        s_col[128 + 2 * lane + 1] = t.c[3];
        const int cw = C < XCH ? C : XCH;
        lc = cw <= 1 ? 0 : cw <= 2 ? 1 : cw <= 4 ? 2 : 3;
        lm = 4 - lc;
        const int s = lane >> lc;
        q = lane & ((1 << lc) - 1);
        w = s >> lm;
        tb = 2 * (((w >> 1) << lm) + (s & ((1 << lm) - 1))) + (w & 1);
        wave_sync();
    }
    // Issues the loads of chunks [c0, c0 + cg) of every item (pair() waits
    // for them when it first reads the pass).
    __device__ __forceinline__ void stage(const double *__restrict__ x, int ks, int c0, int cg)
    {
        const int Cm = (1 << lc) - 1;
        wave_sync();                               // earlier reads of buf are done
        const int n = 4 << lc;                     // a multiple of 4
#pragma unroll 4
        for (int i = 0; i < n; ++i) {
            const int c = (q - 2 * i - (w >> 1)) & Cm;
            if (c < cg) {
                const int cl = s_col[tb + (i << (lm + 2))];
                load_lds16(x + (long long)cl * ks + 2 * (c0 + c), buf + 1024 * i);
            }
        }
    }
    // The x values of pair rr (k even) for this lane's S = 4 items.  The
    // tile's first pass is issued at the top of the tile (so its loads are in
    // flight during the tile's flag and row work); later passes when their
    // first pair is reached.
    __device__ __forceinline__ void pair(const double *__restrict__ x, int ks, int k, int rr,
                                         int lane, double2v (&d)[4])
    {
        const int C = k >> 1, c0 = rr >> 1, cl = c0 % XCH;
        if (cl == 0) {
            if (c0 > 0) stage(x, ks, c0, min(C - c0, XCH));
            lds_dma_wait();
        }
        const int Cm = (1 << lc) - 1, Mm = (1 << lm) - 1;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const int u = (kk >> 1) * 64 + lane;   // item t = 2u + (kk & 1)
            const int r = u & Mm, v = u >> lm;
            const int e = 2 * v + (kk & 1);
            const int s = r + ((e & 3) << lm);
            const int l = (s << lc) + ((cl + v) & Cm);
            d[kk] = *reinterpret_cast<const double2v *>(buf + 1024 * (e >> 2) + 16 * l);
        }
    }
};

// A tile's products (one value or a pair of right-hand sides each) through LDS:
// written as loaded, G consecutive items per lane and load group, read back
// lane-contiguous, item k of lane l being item l*S + k of the tile.
template <typename T, int S, typename V>
__device__ __forceinline__ void tile_transpose(V *sb, const V (&prod)[S], V (&pc)[S], int lane)
{
    constexpr int G = Tile<T, S>::G;
    if constexpr (S == G) {                      // loaded lane-contiguous
#pragma unroll
        for (int k = 0; k < S; ++k) pc[k] = prod[k];
        return;
    }
    constexpr int N = 16 / (int)sizeof(V);       // items per 16-byte unit
    constexpr int U = S / N, H = G / N;          // units per lane, per lane and load group
    typedef unsigned int bits_t __attribute__((ext_vector_type(4)));
    bits_t *su = reinterpret_cast<bits_t *>(sb);
#pragma unroll
    for (int j = 0; j < S / G; ++j)
#pragma unroll
        for (int h = 0; h < H; ++h) {
            bits_t b;
            __builtin_memcpy(&b, &prod[j * G + h * N], 16);
            const int u = lane * H + h;
            const int term = swizzle_term<U>(u) ^ swizzle_term<U>(j * kWave * H);
            su[j * kWave * H + (u ^ term)] = b;
        }
    wave_sync();
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const bits_t b = su[lane * U + (j ^ swizzle_term<U>(lane * U))];
        __builtin_memcpy(&pc[j * N], &b, 16);
    }
    wave_sync();
}

// Lane-sequential segmented sums of a lane's items: at every head (bit k of hb:
// item k starts a row) the sum before it is closed into sb, the lane's first one
// at the place of the segment that the lanes before it leave open (lane 0, whose
// item 0 always starts a segment, has none).  Returns the sum left open.
template <typename V, int S>
__device__ __forceinline__ V lane_segments(V *sb, const V (&pc)[S], unsigned hb, int seg_base,
                                           int lane, V zero)
{
    V acc = zero;
    int sidx = lane == 0 ? -1 : seg_base - 1;
#pragma unroll
    for (int kk = 0; kk < S; ++kk) {
        const int h = __builtin_amdgcn_sbfe((int)hb, kk, 1);   // -1 at a head
        if (kk == 0) {
            if (h && lane > 0) sb[sidx] = zero;
        } else if (h) {
            sb[sidx] = acc;
        }
        sidx -= h;
        acc = zero_where(acc, h);
        acc += pc[kk];
    }
    return acc;
}

template <int R>
struct RhsTag {
    static constexpr int value = R;
};

// XCH > 0 (fp64, S = 4, KMAX > 1): right-hand-side pairs take their x values
// from the tile staged in LDS, XCH chunks per item at a time (XStage), at
// s_stage: 1 KB of column indices, then the staging buffer.
// NOEMPTY: the matrix has no empty rows (the stacked matrix of the column-panel
// layout), so no tile is dirty and the empty-row paths are left out.
template <typename T, int S, int KMAX, bool STRIDED, bool STATS, int CP, int XCH = 0,
          bool NOEMPTY = false>
__device__ __forceinline__ void segsum_wave(const MatView<T> &mv, const int w, const int lane,
                                            unsigned *s_head, T *s_buf, T *s_carry, const T alpha,
                                            unsigned long long *stats,
                                            unsigned char *s_stage = nullptr, int touch = 0)
{
    constexpr int P = kWave * S;
    constexpr int G = Tile<T, S>::G;
    const int k = (KMAX == 1) ? 1 : mv.k;
    const int ks = STRIDED ? mv.kstride : 1;
    // right-hand sides in pairs: k even at an even stride, from x and y
    // offsets that keep the 2-wide loads and stores aligned; only where a
    // tile's pairs fit the registers (S * sizeof(T) <= 32 bytes per lane)
    constexpr bool kPairs = KMAX > 1 && S * sizeof(T) <= 32;
    const bool pairs = kPairs && (ks & 1) == 0 && (k & 1) == 0;
    constexpr bool kStage = XCH > 0 && kPairs && std::is_same<T, double>::value && S == 4;
    [[maybe_unused]] XStage<(XCH > 0 ? XCH : 1)> xs{kStage ? s_stage + 1024 : nullptr,
                                                   reinterpret_cast<int *>(s_stage)};
    const int *__restrict__ row_ptr = mv.row_ptr;
    const int *__restrict__ tile_row = mv.tile_row;
    const T *__restrict__ x = mv.x;
    T *__restrict__ y = mv.y;

    // Rows before the first nonzero belong to no tile: spread their zeroing.
    if (!NOEMPTY && mv.lead_empty > 0) {
        const long long lo = (long long)mv.lead_empty * w / mv.NW;
        const long long hi = (long long)mv.lead_empty * (w + 1) / mv.NW;
        for (long long r = lo + lane; r < hi; r += kWave)
            for (int rr = 0; rr < k; ++rr) y[r * ks + rr] = T(0);
    }

    const int p_begin = w * mv.TPW;
    const int p_end = min(p_begin + mv.TPW, mv.NP);
    const int E0 = p_begin * P;
    const int r_first = tile_row[p_begin];
    bool syncing = false;                       // first row began in an earlier wave
    bool did_sync = false;
    // The wave's one boundary-row partial (KMAX == 1) stays in registers and is
    // stored after the tile loop: a store inside the loop would make the
    // compiler wait for it (and, the counter being in order, for every load
    // issued since) before its data register is reused.
    int sync_key = -1;
    T sync_v1 = T(0);
    bool open = false;                          // a row continues past the last tile
    T carry1 = T(0);                            // the open row's partial (KMAX == 1)
    if (KMAX > 1) {
        if (lane < k) s_carry[lane] = T(0);
        wave_sync();
    }
    auto carry_get = [&](int rr) -> T {
        if constexpr (KMAX == 1) return carry1;
        else return s_carry[rr];
    };
    // the open row's partial of RHS rr .. rr+R-1 as a value (R = 1) or pair
    auto carry_getv = [&](auto rt, int rr) {
        constexpr int R = decltype(rt)::value;
        using V = typename RhsVec<T, R>::type;
        if constexpr (R == 1) return carry_get(rr);
        else return *reinterpret_cast<const V *>(s_carry + rr);
    };
    auto carry_setv = [&](auto rt, int rr, typename RhsVec<T, decltype(rt)::value>::type v) {
        constexpr int R = decltype(rt)::value;
        using V = typename RhsVec<T, R>::type;
        if constexpr (KMAX == 1) carry1 = v;
        else {
            if (lane == 0) *reinterpret_cast<V *>(s_carry + rr) = v;
            wave_sync();
        }
    };
    unsigned long long n_fast = 0, n_dirty = 0;

    // Row chunk of the next tile loaded one tile ahead.  The next tile's
    // stream is in flight while this one is reduced (kPrefetch) in fp32 and with
    // several right-hand sides.  In fp64 with one right-hand side a tile is
    // loaded at the top of its own iteration: there the prefetched tile holds
    // 24 more VGPRs, and the four-panel power-law tiles ran 0.4-1.9 us slower
    // with it (fp32 0.6 us faster, the plain and banded tiles alike).
    constexpr bool kPrefetch = KMAX > 1 || sizeof(T) < 8;
    Tile<T, S> cur;
    tile_load<T, S>(mv.col, mv.val, E0, lane, cur);
    constexpr int CR = CP * kWave;              // rows a chunk covers
    RowChunk<CP> rc = load_chunk<CP>(row_ptr, r_first, lane, mv.m);
    int r1 = r_first;
    // the caller's read-ahead of x (issued before the loads above) is
    // consumed here, so its register is free during the tile loop
    asm volatile("" ::"v"(touch));   // emits no instruction

    for (int p = p_begin; p < p_end; ++p) {
        const int B = p * P;
        const int r0 = r1;
        r1 = tile_row[p + 1];
        const bool general = r0 != r1;
        if constexpr (!kPrefetch) {
            if (p != p_begin) tile_load<T, S>(mv.col, mv.val, B, lane, cur);
        }
        RhsX<T, S, KMAX> xr;
        [[maybe_unused]] RhsPair<T, S> xp;
        if constexpr (kStage) {
            if (pairs) {
                xs.begin_tile(cur, lane, k >> 1);
                xs.stage(x, ks, 0, min(k >> 1, XCH));   // waited for by the first pair
            } else {
                xr.first(x, cur, ks);
            }
        } else if constexpr (kPairs) {
            if (pairs) xp.first(x, cur, ks);
            else xr.first(x, cur, ks);
        } else {
            xr.first(x, cur, ks);
        }
        const RowChunk<CP> cc = rc;
        if (p + 1 < p_end) rc = load_chunk<CP>(row_ptr, r1, lane, mv.m);
        __builtin_amdgcn_sched_barrier(0);
        [[maybe_unused]] Tile<T, S> nxt;
        if (kPrefetch && p + 1 < p_end)           // wave-uniform; the last tile loads nothing more
            tile_load<T, S>(mv.col, mv.val, B + P, lane, nxt);

        const bool cont = read_lane(cc.a[0], 0) < B;   // item 0 continues row r0 (lane 0 holds row r0)
        if (p == p_begin) syncing = cont;
        const bool tail = B + P > mv.nnz;

        // products of the tile for RHS rr .. rr+R-1 (items past nnz masked)
        auto products = [&](auto rt, const auto &xv, auto (&prod)[S]) {
#pragma unroll
            for (int kk = 0; kk < S; ++kk) {
                const auto pk = cur.v[kk] * xv[kk];
                prod[kk] = tail ? keep_or_zero(pk, tile_item<T, S>(B, lane, kk) < mv.nnz) : pk;
            }
        };
        if (!general) {                          // fast track
            auto fast_rhs = [&](auto rt, int rr, const auto &xv) __attribute__((always_inline)) {
                using V = typename RhsVec<T, decltype(rt)::value>::type;
                V prod[S];
                products(rt, xv, prod);
                V s = prod[0];
#pragma unroll
                for (int kk = 1; kk < S; ++kk) s += prod[kk];
                s = wave_sum(s);
                carry_setv(rt, rr, cont ? carry_getv(rt, rr) + s : s);
            };
            bool done = false;
            if constexpr (kStage) {
                if (pairs) {
                    for (int rr = 0; rr < k; rr += 2) {
                        double2v xv[4];
                        xs.pair(x, ks, k, rr, lane, xv);
                        fast_rhs(RhsTag<2>{}, rr, xv);
                    }
                    done = true;
                }
            } else if constexpr (kPairs) {
                if (pairs) {
                    for (int rr = 0; rr < k; rr += 2) {
                        xp.issue(x, cur, ks, rr, k);
                        fast_rhs(RhsTag<2>{}, rr, xp.v);
                        xp.advance(rr, k);
                    }
                    done = true;
                }
            }
            if (!done)
                for (int rr = 0; rr < k; ++rr) {
                    xr.issue(x, cur, ks, rr, k);
                    fast_rhs(RhsTag<1>{}, rr, xr.v);
                    xr.advance(rr, k);
                }
            open = true;
            if (STATS) ++n_fast;
        } else {
            // A tile of fewer than CR rows takes every row boundary from
            // its chunk; only longer tiles load more row_ptr values, in
            // loops.  The two cases are separate instantiations, so the loops
            // (and the waits they need) are not on the common path at all.
            auto general_tile = [&](auto big) __attribute__((always_inline)) {
                constexpr bool BIG = decltype(big)::value;
                // ---- bit flags (once for all right-hand sides) ------------------
                const int stop = (r1 == mv.m) ? mv.m - 1 : r1;
                // nonempty rows of the chunk, one ballot per 64 rows (kept as
                // wave-wide masks, not per-lane registers, until the output)
                uint64_t mne[CP];
                bool lane_dirty = false;
                wave_sync();                         // previous tile's LDS reads are done
                s_head[lane] = 0u;
                wave_sync();
                // (empty rows of the chunk get their zero in the output step,
                // after this tile's loads have been consumed)
                static_for<CP>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    mne[q] = 0ull;
                    if (q > 0 && r0 + q * kWave > stop) return;   // wave-uniform: no rows here
                    // the shift reads the next lane: it runs on the whole
                    // wave, before any lane-dependent condition masks lanes off
                    const bool have = r0 + q * kWave + lane <= stop;
                    bool ne = have;
                    if constexpr (!NOEMPTY) ne = have && chunk_next<q>(cc, lane) > cc.a[q];
                    lane_dirty = lane_dirty || (have && !ne);
                    mne[q] = ballot(ne);
                    if (ne) {
                        const int o = cc.a[q] - B;
                        if (o >= 0 && o < P) atomicOr(&s_head[o / S], 1u << (o % S));
                    }
                });
                if constexpr (BIG)
                for (int rb = r0 + CR; rb <= stop;) {   // >= CR rows
                    const int rq = min(rb + lane, stop);
                    const int rp = row_ptr[rq];
                    if constexpr (NOEMPTY) {
                        if (rb + lane <= stop) {
                            const int o = rp - B;
                            if (o >= 0 && o < P) atomicOr(&s_head[o / S], 1u << (o % S));
                        }
                        rb += kWave;
                        continue;
                    }
                    const int rpn = row_ptr[rq + 1];
                    const int vb = row_ptr[min(rb + kWave, stop + 1)];
                    if (rb + kWave <= stop && read_lane(rp, 0) == vb) {
                        // 64 empty rows with more rows after them: skip the whole run
                        const int re = empty_run_end(row_ptr, rb + kWave, vb, stop);
                        lane_dirty = true;
                        zero_run(y, (long long)rb * ks, (long long)re * ks, lane);
                        rb = re;
                        continue;
                    }
                    if (rb + lane <= stop) {
                        if (rpn > rp) {
                            const int o = rp - B;
                            if (o >= 0 && o < P) atomicOr(&s_head[o / S], 1u << (o % S));
                        } else {
                            lane_dirty = true;
                            for (int rr = 0; rr < k; ++rr) y[(long long)(rb + lane) * ks + rr] = T(0);
                        }
                    }
                    rb += kWave;
                }
                const bool dirty = !NOEMPTY && ballot(lane_dirty) != 0ull;
                wave_sync();
                unsigned hb = s_head[lane];
                if (lane == 0) hb |= 1u;

                // ---- segment numbers -----------------------------------------
                const int nh = __popc(hb);
                const int incl = wave_incl_scan(nh, lane);
                const int seg_base = incl - nh;
                const int K = read_lane(incl, kWave - 1);
                // row_ptr[r1] sits in the chunk when r1 < r0+CR
                int rp_r1;
                if (!BIG || r1 - r0 < CR) {
                    // read the lane out of every part, then pick one: a
                    // select among registers by a run-time index would be
                    // compiled as an indexed load from scratch memory
                    const int d = r1 - r0, q = d / kWave, l = d % kWave;
                    rp_r1 = read_lane(cc.a[0], l);
                    static_for<CP>([&](auto qc) {
                        if constexpr (decltype(qc)::value > 0) {
                            const int v = read_lane(cc.a[qc], l);
                            if (q == qc) rp_r1 = v;
                        }
                    });
                } else {
                    rp_r1 = row_ptr[min(r1, mv.m)];
                }
                const bool partial_tail = (r1 < mv.m) && (rp_r1 < B + P);
                const int kb = syncing ? 1 : 0;
                const int ke = partial_tail ? K - 1 : K;

                if (STATS && dirty) ++n_dirty;

                auto general_rhs = [&](auto rt, int rr, const auto &xv) __attribute__((always_inline)) {
                    constexpr int R = decltype(rt)::value;
                    using V = typename RhsVec<T, R>::type;
                    V *sb = reinterpret_cast<V *>(s_buf);
                    const V zero = static_cast<V>(T(0));
                    auto store_y = [&](long long row, V val) {
                        *reinterpret_cast<V *>(y + row * ks + rr) = val;
                    };
                    V prod[S];
                    products(rt, xv, prod);
                    // products -> LDS in tile order, back lane-contiguous
                    wave_sync();
                    V pc[S];
                    tile_transpose<T, S>(sb, prod, pc, lane);
                    if (lane == 0 && cont) pc[0] = pc[0] + carry_getv(rt, rr);

                    // ---- lane-sequential segmented reduction -----------------
                    const V acc = lane_segments(sb, pc, hb, seg_base, lane, zero);

                    // ---- segments spanning lanes -----------------------------
                    const uint64_t present = ballot(hb != 0u);   // bit 0 always set
                    const V I = wave_segscan(acc, present, lane);
                    const V Iprev = dpp<kDppWaveShr1>(I);     // lane i <- lane i-1 (lane 0: unused)
                    if (hb && lane > 0) sb[seg_base - 1] = Iprev + sb[seg_base - 1];
                    if (lane == kWave - 1) sb[K - 1] = I;
                    wave_sync();

                    // ---- output ------------------------------------------------
                    if (!dirty) {
                        for (int kk = kb + lane; kk < ke; kk += kWave)
                            store_y(r0 + kk, alpha * sb[kk]);
                    } else {
                        // a nonempty row's segment is its rank among the
                        // tile's nonempty rows; an empty row gets 0
                        int running = 0;
                        static_for<CP>([&](auto qc) {
                            constexpr int q = decltype(qc)::value;
                            if (q > 0 && r0 + q * kWave > stop) return;   // wave-uniform
                            const int row = r0 + q * kWave + lane;
                            const bool ne = (mne[q] >> lane) & 1ull;
                            const int rank = running + popc_below(mne[q]);
                            if (ne && rank >= kb && rank < ke)
                                store_y(row, alpha * sb[rank]);
                            else if (row <= stop && !ne)
                                store_y(row, zero);
                            running += __popcll(mne[q]);
                        });
                        if constexpr (BIG)
                        for (int rb = r0 + CR; rb <= stop;) {   // >= CR rows
                            const int rq = min(rb + lane, stop);
                            const int rp = row_ptr[rq], rpn = row_ptr[rq + 1];
                            const int vb = row_ptr[min(rb + kWave, stop + 1)];
                            if (rb + kWave <= stop && read_lane(rp, 0) == vb) {
                                rb = empty_run_end(row_ptr, rb + kWave, vb, stop);   // no segments
                                continue;
                            }
                            const int r = rb + lane;
                            const bool ne = r <= stop && rpn > rp;
                            const uint64_t msk = ballot(ne);
                            const int rank = running + popc_below(msk);
                            if (ne && rank >= kb && rank < ke)
                                store_y(r, alpha * sb[rank]);
                            running += __popcll(msk);
                            rb += kWave;
                        }
                    }
                    if (syncing) {
                        if constexpr (KMAX == 1) sync_v1 = alpha * s_buf[0];
                        else if (lane == 0)
                            *reinterpret_cast<V *>(mv.sync_val + (long long)w * KMAX + rr) =
                                alpha * sb[0];
                    }
                    carry_setv(rt, rr, sb[K - 1]);
                };
                bool done = false;
                if constexpr (kStage) {
                    if (pairs) {
                        for (int rr = 0; rr < k; rr += 2) {
                            double2v xv[4];
                            xs.pair(x, ks, k, rr, lane, xv);
                            general_rhs(RhsTag<2>{}, rr, xv);
                        }
                        done = true;
                    }
                } else if constexpr (kPairs) {
                    if (pairs) {
                        for (int rr = 0; rr < k; rr += 2) {
                            xp.issue(x, cur, ks, rr, k);
                            general_rhs(RhsTag<2>{}, rr, xp.v);
                            xp.advance(rr, k);
                        }
                        done = true;
                    }
                }
                if (!done)
                    for (int rr = 0; rr < k; ++rr) {
                        xr.issue(x, cur, ks, rr, k);
                        general_rhs(RhsTag<1>{}, rr, xr.v);
                        xr.advance(rr, k);
                    }
                if (syncing) {
                    sync_key = mv.key_base + r0 * ks;
                    syncing = false;
                    did_sync = true;
                }
                open = partial_tail;
                // the long-tile path ends with nothing in flight, so registers
                // its row_ptr loads used carry no pending write into the next
                // tile (which would otherwise wait for every load in flight)
                if constexpr (BIG) __builtin_amdgcn_s_waitcnt(0);
            };
            if (r1 - r0 < CR) general_tile(BigTag<false>{});
            else general_tile(BigTag<true>{});
        }
        if constexpr (kPrefetch) cur = nxt;
    }

    if (open) {
        const int r_open = tile_row[p_end];
        if (syncing) {
            sync_key = mv.key_base + r_open * ks;
            if constexpr (KMAX == 1) sync_v1 = alpha * carry_get(0);
            else if (lane == 0)
                for (int rr = 0; rr < k; ++rr)
                    mv.sync_val[(long long)w * KMAX + rr] = alpha * carry_get(rr);
            did_sync = true;
        } else if (lane == 0) {
            for (int rr = 0; rr < k; ++rr) y[(long long)r_open * ks + rr] = alpha * carry_get(rr);
        }
    }
    if (lane == 0) {
        mv.sync_row[w] = did_sync ? sync_key : -1;
        if (KMAX == 1 && did_sync) mv.sync_val[w] = sync_v1;
    }
    if (STATS && lane == 0) {
        atomicAdd(&stats[0], n_fast);
        atomicAdd(&stats[1], n_dirty);
        atomicAdd(&stats[2], did_sync ? 1ull : 0ull);
    }
}

template <typename T, int S, bool STATS, int CP, bool NOEMPTY = false>
__global__ __launch_bounds__(512) void segsum_kernel(
    const int *__restrict__ row_ptr, const int *__restrict__ col, const T *__restrict__ val,
    const T *__restrict__ x, T *__restrict__ y, const int *__restrict__ tile_row,
    int *__restrict__ sync_row, T *__restrict__ sync_val, unsigned long long *__restrict__ stats,
    const SegsumParams<T> q)
{
    extern __shared__ double smem_raw[];
    const int lane = lane_id();
    // q.x_lines > 0 (x small enough for every L2): the blocks of each XCD
    // (dealt round-robin, block b on XCD b % 8) read one word of every
    // 128-byte line of x between them, so the first tile's gathers hit L2.
    int touch = 0;
    {
        const long long t = (long long)(blockIdx.x / 8) * blockDim.x + threadIdx.x;
        if (t < q.x_lines) touch = reinterpret_cast<const int *>(x)[t * (128 / sizeof(int))];
    }
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int blk = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int w = blk * q.wpb + wib;
    if (w >= q.NW) return;
    unsigned char *wave_lds = reinterpret_cast<unsigned char *>(smem_raw) + wib * q.wave_lds_bytes;
    MatView<T> mv{row_ptr, tile_row, col, val, x, y, sync_row, sync_val,
                  q.m, q.nnz, q.NP, q.NW, q.lead_empty, 1, 1, q.TPW, 0};
    segsum_wave<T, S, 1, false, STATS, CP, 0, NOEMPTY>(
        mv, w, lane, reinterpret_cast<unsigned *>(wave_lds),
        reinterpret_cast<T *>(wave_lds + 256), nullptr, q.alpha, stats, nullptr, touch);
}

// ---------------------------------------------------------------------------
// One wave per tile: the sums of segsum_wave, bit for bit, with the TPW tiles
// of a logical wave spread over TPW neighbouring waves of one block.
//
// The tile loop runs a logical wave's tiles one after the other because the
// open row's partial passes from each to the next.  But only the first segment
// of a tile needs that partial, so here every wave loads, multiplies and reduces
// its own tile at once, leaves its closing sum in LDS, and after one barrier
// takes the partial from the tiles before it and redoes that one segment, in the
// order of the loop.  A matrix of few logical waves then has TPW times as many
// waves to hide its loads behind (65,536 uniform rows at the default tile, 513
// logical waves: 14.0 -> 8.2 us in the kernel; 8,000 nonzeros: 10.0 -> 5.5).
//
// On large matrices the loop's registers (100 in fp64 at S = 8: 4 waves per
// SIMD, 58 here: 8) were not the bound, its instructions and LDS conflicts were
// part of it: counters on the 3x3-block matrix (fp32, 54M nonzeros) put the
// vector ALU at 31%, the LDS at 30% (71% of it bank conflicts of the product
// transpose) and the texture address units at 84% of the time.  So products go
// to LDS swizzled (swizzle_term: no conflicts left, LDS at 10%), the lane-sequential
// reduction has one masked LDS store per item and no other branch, the scan
// takes its lane conditions from scalar masks, and gathers use 32-bit offsets.
// Default tile, call with caches warm, fp64: 7-point Laplacian 160^3 91 -> 80 us,
// 3x3 blocks 160 -> 154, power law (whose gathers miss L2) 119 -> 114.
// What is left there is memory: 424 MB in 78 us is 5.4 TB/s.  Tried on top and
// slower: G neighbouring x values per lane in one wide load where columns run on
// (3x3 blocks fp64 153 -> 170 us: the unit's time is the lines, not the
// accesses); consecutive items on consecutive lanes (Laplacian fp32 58 -> 62);
// fewer waves per CU through more LDS (Laplacian 82 -> 90).
// ---------------------------------------------------------------------------
constexpr int kMaxGroup = 8;   // waves of a block, and the largest tiles_per_wave

// What the waves of a block hand to each other: every tile's closing sum and
// its kind (bit 0: inside one row, bit 1: its first item continues a row).
template <typename T>
struct TileShare {
    T val[kMaxGroup];
    int kind[kMaxGroup];
};

// Rows that cross logical waves, finished inside the launch.  The waves
// first..last holding one row's nonzeros each send a partial; whoever comes
// last adds them up, in the order of calibrate_window (wave order within
// windows of 64 waves, then the first wave's own partial), and stores y.
// Nobody waits for a wave that has not run.  Words are tagged with the call's
// number, so that anything another call left behind reads as empty, and are set
// back to 0 by the wave that finishes the row, so that a replay of the same
// call starts empty too.  They are written through to, and read from, the
// point where the eight L2s meet (agent scope).
struct ChainBuf {
    unsigned long long *pair;    // [NW * sizeof(T)/4] rows of two waves, by first wave
    unsigned long long *count;   // [NW] call << 32 | arrivals, by first wave (of a row, of a group)
    void *own, *part;            // [NW] T: longer rows, the first wave's partial and the others'
    unsigned call;               // the call's number, 1 .. 2^31 - 1
};

template <typename U>
__device__ __forceinline__ U agent_load(const U *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ __forceinline__ void agent_store(U *p, U v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether this is the last of n > 1 arrivals at `word`: the first one sets the tag
// there, the rest add to it.
__device__ __forceinline__ bool chain_arrive(unsigned long long *word, unsigned tag, int n)
{
    unsigned long long seen = 0ull;
    while (seen >> 32 != tag)
        if (__hip_atomic_compare_exchange_strong(word, &seen, (unsigned long long)tag << 32 | 1ull,
                                                 __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return false;
    return (unsigned)__hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT) == (unsigned)n - 1;
}

// Waves up to which a row's partials are counted at one word, and of a group
// beyond.  A word takes an arrival every 28 ns or so: one row over 390 (800)
// logical waves among 500,000 nonzeros, fp64, S = 4, T = 1, 14.6 (24.9) us a call
// with one word, 8.0 (8.3) with groups, 9.7 (13.6) with calibrate_kernel.
constexpr int kChainDirect = 64, kChainGroup = 32;

// Wave w's partial v of `row`, whose nonzeros lie in waves first..last > first.
template <typename T>
__device__ __forceinline__ void chain_add(const ChainBuf &cb, int row, int first, int last, int w,
                                          T v, int lane, T *__restrict__ y)
{
    constexpr int H = sizeof(T) / 4;             // 32-bit halves of a partial
    const int e0 = first + 1, base = e0 & ~(kWave - 1);
    const int end = min(last - base, kWave - 1);
    if (last == e0) {
        // Two waves swap: lane h exchanges {tag, half h} for what lies there.
        // The one that finds both of the other's halves finishes the row.  Were the
        // halves swapped in different orders, each wave finds one; both then
        // exchange the count, and the second to do so has the half that it
        // lacks in memory: the other wave's exchanges are over.
        const unsigned tag = cb.call << 1 | (w == first ? 0u : 1u);   // the two sides differ
        unsigned half;
        if constexpr (H == 2) {
            const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
            half = (unsigned)(lane == 0 ? b : b >> 32);
        } else {
            half = __builtin_bit_cast(unsigned, v);
        }
        unsigned long long *p = cb.pair + (long long)first * H + lane;
        unsigned long long got = 0ull;
        if (lane < H)
            got = __hip_atomic_exchange(p, (unsigned long long)tag << 32 | half, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
        const bool found = (unsigned)(got >> 32) == (tag ^ 1u);   // no call's tag is 0
        const uint64_t halves = ballot(found);
        if (halves == 0) return;
        if constexpr (H == 2) {
            if (halves != 3) {
                unsigned long long seen = 0ull;
                if (lane == 0)
                    seen = __hip_atomic_exchange(cb.count + first,
                                                 (unsigned long long)cb.call << 32 | 1ull,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (__builtin_amdgcn_readfirstlane((unsigned)(seen >> 32)) != cb.call) return;
                if (lane < H && !found) got = agent_load(p);
                if (lane == 0) agent_store(cb.count + first, 0ull);
            }
        }
        const unsigned lo = (unsigned)read_lane((int)(unsigned)got, 0);
        T o;
        if constexpr (H == 2) {
            const unsigned hi = (unsigned)read_lane((int)(unsigned)got, 1);
            o = __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
        } else {
            o = __builtin_bit_cast(float, lo);
        }
        const T head = w == first ? v : o;
        T tot = w == first ? o : v;
        if (end == kWave - 1) tot = tot + T(0);       // as at a window's last entry
        if (lane == 0) y[row] = head + tot;
        // last: a store ahead of a use of `got` would be waited for there
        if (lane < H) agent_store(p, 0ull);
        return;
    }
    T *own = reinterpret_cast<T *>(cb.own), *part = reinterpret_cast<T *>(cb.part);
    // Groups are counted at their first wave's word (no other row's: this one goes
    // on past that wave, or the group is that wave alone and is not counted), and
    // the groups at the row's pair word, free in a row of more than two waves.
    int complete = 0;
    if (lane == 0) {
        agent_store(w == first ? own + first : part + w, v);
        // the partial has arrived before the count says so
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const int n = last - first + 1;
        if (n <= kChainDirect) {
            complete = chain_arrive(cb.count + first, cb.call, n);
        } else {
            const int g = w & ~(kChainGroup - 1), g0 = max(first, g);
            const int ng = min(last, g + kChainGroup - 1) - g0 + 1;
            complete = ng == 1 || chain_arrive(cb.count + g0, cb.call, ng);
            if (complete) {
                if (ng > 1) agent_store(cb.count + g0, 0ull);
                complete = chain_arrive(cb.pair + (long long)first * H, cb.call << 1,
                                        last / kChainGroup - first / kChainGroup + 1);
            }
        }
        asm volatile("" ::: "memory");
    }
    if (!__builtin_amdgcn_readfirstlane(complete)) return;
    const int e = base + lane;
    const bool on = e >= e0 && e <= last;
    const T pv = on ? agent_load(part + e) : T(0);
    T tot = read_lane(wave_segscan(pv, 1ull << (e0 - base) | 1ull, lane), end);
    if (end == kWave - 1) {                 // up to a window's last entry: later windows follow
        T ext = T(0);
        for (int nb = base + kWave; nb <= last; nb += 4 * kWave) {   // four windows on their way at once
            T pn[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int e = nb + i * kWave + lane;
                pn[i] = e <= last ? agent_load(part + e) : T(0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (nb + i * kWave <= last) ext = ext + wave_sum(pn[i]);
        }
        tot = tot + ext;
    }
    if (lane == 0) {
        const T head = w == first ? v : agent_load(own + first);
        y[row] = head + tot;
        agent_store(last - first < kChainDirect ? cb.count + first : cb.pair + (long long)first * H,
                    0ull);
    }
}

// The last row r >= lo with row_ptr[r] <= key, given row_ptr[lo] = vlo <= key.
// A round cuts the bracket into 17 parts (16 probes: 64 would need a round less,
// but each is a cache line, and the line rate from L2 is what gathers wait for:
// power law, 10M nonzeros, fp32, 73.6 us a call with 64, 68.4 with 16 or 8), then
// reads the 256 rows around the place where rows of even length would put key.
// Between even rows that finds it at once; otherwise the bracket has shrunk.  `guesses`: rounds at the start that read the 256 rows only (two where
// even_rows says so: a stencil's border rows put the first guess off by some
// thousand rows, and the second, from the edge of the first, right).
__device__ __forceinline__ int find_row(const int *__restrict__ row_ptr, int m, int nnz, int key,
                                        int lo, int vlo, int guesses, int lane)
{
    constexpr int W = 4 * kWave, kProbes = 16;
    int hi = m + 1, vhi = nnz;             // row_ptr[hi] > key (past the end at first)
    for (;; --guesses) {
        if (guesses <= 0 && hi - lo > W) {
            const int i = min(lane, kProbes - 1) + 1;
            const int at = lo + (int)((long long)(hi - lo) * i / (kProbes + 1));
            const int v = row_ptr[at];
            const int n = __popcll(ballot(v <= key && lane < kProbes));   // a prefix of the lanes
            if (n < kProbes) hi = read_lane(at, n), vhi = read_lane(v, n);
            if (n > 0) lo = read_lane(at, n - 1), vlo = read_lane(v, n - 1);
        }
        int g = lo;
        if (hi - lo > W) {
            const float f = (float)(key - vlo) / (float)max(vhi - vlo, 1) * (float)(hi - lo);
            g = __builtin_amdgcn_readfirstlane(lo + (int)f) - W / 2;
            g = max(lo, min(g, hi - W));
        }
        // rows [g, g + W) of the bracket; the whole bracket if it is no longer
        int v[4], n = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = row_ptr[min(g + q * kWave + lane, m)];
#pragma unroll
        for (int q = 0; q < 4; ++q) n += __popcll(ballot(g + q * kWave + lane < hi && v[q] <= key));
        if (hi - lo <= W || (n > 0 && n < W)) return g + n - 1;
        if (n == 0) hi = g, vhi = read_lane(v[0], 0);
        else lo = g + W - 1, vlo = read_lane(v[3], kWave - 1);
    }
}

// Whether the middle row starts within 128 rows of where rows of even length
// would put it (bands, stencils, dense blocks; hardly ever a power law).
__device__ __forceinline__ bool even_rows(const int *__restrict__ row_ptr, int m, int nnz)
{
    const int h = m >> 1;
    const float per = (float)nnz / (float)m;
    return fabsf((float)row_ptr[h] - per * (float)h) < 128.0f * per;
}

// BOUNDED: col/val hold exactly nnz items (no padding), so a tile reaching
// past nnz is loaded with checked indices (a wave-uniform branch).  SEARCH: no
// tile_row; each wave finds its first row (while its stream is on its way) and
// its last from the row chunk.  FUSED: rows crossing logical waves are finished
// here (chain_add), else their partials are left to calibrate_kernel.
template <typename T, int S, int CP, bool BOUNDED, bool SEARCH, bool FUSED>
__global__ __launch_bounds__(512) void segsum_tiles_kernel(
    const int *__restrict__ row_ptr, const int *__restrict__ col, const T *__restrict__ val,
    const T *__restrict__ x, T *__restrict__ y, const int *__restrict__ tile_row,
    int *__restrict__ sync_row, T *__restrict__ sync_val, const ChainBuf cb,
    const SegsumParams<T> q)
{
    constexpr int P = kWave * S;
    constexpr int CR = CP * kWave;
    extern __shared__ double smem_raw[];
    const int lane = lane_id();
    int touch = 0;
    {
        const long long t = (long long)(blockIdx.x / 8) * blockDim.x + threadIdx.x;
        if (t < q.x_lines) touch = reinterpret_cast<const int *>(x)[t * (128 / sizeof(int))];
    }
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwb = blockDim.x >> 6;
    const int p = xcd_remap((int)blockIdx.x, (int)gridDim.x) * nwb + wib;
    const int TPW = q.TPW;                      // a power of two
    const int g0 = wib & ~(TPW - 1);            // the logical wave's first tile in the block
    const int w = p >> __builtin_ctz(TPW);
    // product buffers first (16-byte aligned), then the head words, then the hand-over
    T *sb = reinterpret_cast<T *>(smem_raw) + wib * P;
    unsigned *s_head = reinterpret_cast<unsigned *>(reinterpret_cast<T *>(smem_raw) + nwb * P) +
                       wib * kWave;
    TileShare<T> &sh = *reinterpret_cast<TileShare<T> *>(
        reinterpret_cast<unsigned *>(reinterpret_cast<T *>(smem_raw) + nwb * P) + nwb * kWave);
    const bool active = p < q.NP;
    const int pe = active ? p : 0;
    const int B = pe * P;
    const T alpha = q.alpha;

    Tile<T, S> t;
    if (BOUNDED && B + P > q.nnz) tile_load_checked<T, S>(col, val, B, lane, q.nnz, t);
    else tile_load<T, S>(col, val, B, lane, t);
    int r0, r1;
    if constexpr (SEARCH) {
        const int guesses = even_rows(row_ptr, q.m, q.nnz) ? 2 : 0;
        r0 = find_row(row_ptr, q.m, q.nnz, B, 0, 0, guesses, lane);
    } else {
        r0 = tile_row[pe];
        r1 = active ? tile_row[pe + 1] : r0;
    }
    const RowChunk<CP> cc = load_chunk<CP>(row_ptr, r0, lane, q.m);
    __builtin_amdgcn_sched_barrier(0);
    T prod[S];
    {
        T xv[S];
        if (q.x_far) {
#pragma unroll
            for (int k = 0; k < S; ++k) xv[k] = x[t.c[k]];
        } else {                      // x below 4 GB: 32-bit offsets, one instruction each
#pragma unroll
            for (int k = 0; k < S; ++k)
                xv[k] = *reinterpret_cast<const T *>(reinterpret_cast<const char *>(x) +
                                                     (unsigned)t.c[k] * (unsigned)sizeof(T));
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::"v"(touch));   // emits no instruction
#pragma unroll
        for (int k = 0; k < S; ++k) prod[k] = t.v[k] * xv[k];
        if (B + P > q.nnz) {
#pragma unroll
            for (int k = 0; k < S; ++k)
                prod[k] = keep_or_zero(prod[k], tile_item<T, S>(B, lane, k) < q.nnz);
        }
    }
    if constexpr (SEARCH) {
        // the last row starting at or before the tile's end: count the chunk's
        // starts up to there, and search on only if all of them are
        r1 = r0;
        if (active) {
            const int key = min(B + P, q.nnz);
            int cnt = 0;
            static_for<CP>([&](auto qc) {
                cnt += __popcll(ballot(cc.a[qc] <= key && r0 + qc * kWave + lane <= q.m));
            });
            r1 = r0 + cnt - 1;
            if (cnt == CR)
                r1 = find_row(row_ptr, q.m, q.nnz, key, r1, read_lane(cc.a[CP - 1], kWave - 1), 0,
                              lane);
        }
    }
    // rows before the first nonzero belong to no tile: spread their zeroing
    int lead_empty = q.lead_empty;              // < 0: not known to the host
    if constexpr (SEARCH)
        lead_empty = row_ptr[1] > 0 ? 0 : find_row(row_ptr, q.m, q.nnz, 0, 0, 0, 0, lane);
    else if (lead_empty < 0)
        lead_empty = tile_row[0];
    if (lead_empty > 0 && active) {
        const unsigned n = (unsigned)lead_empty, per = (n + (unsigned)q.NP - 1) / (unsigned)q.NP;
        const unsigned lo = (unsigned)p * per;               // at most n + NP
        for (unsigned r = lo + lane; r < lo + per && r < n; r += kWave) y[r] = T(0);
    }

    const bool general = r0 != r1;
    const int rp_r1 = row_ptr[min(r1, q.m)], rp_next = row_ptr[min(r1 + 1, q.m)];
    const bool cont = read_lane(cc.a[0], 0) < B;   // item 0 continues row r0
    const int stop = (r1 == q.m) ? q.m - 1 : r1;
    const bool big = r1 - r0 >= CR;
    uint64_t mne[CP];
    unsigned hb = 0;
    bool dirty = false, partial_tail = false;
    int seg_base = 0, K = 0;
    T acc = T(0), I = T(0), out_val;
    T pc[S];
    uint64_t present = 1;
    if (general) {
        // ---- bit flags
        bool lane_dirty = false;
        s_head[lane] = 0u;
        wave_sync();
        static_for<CP>([&](auto qc) {
            constexpr int qq = decltype(qc)::value;
            mne[qq] = 0ull;
            if (qq > 0 && r0 + qq * kWave > stop) return;   // wave-uniform: no rows here
            const bool have = r0 + qq * kWave + lane <= stop;
            const bool ne = have && chunk_next<qq>(cc, lane) > cc.a[qq];
            lane_dirty = lane_dirty || (have && !ne);
            mne[qq] = ballot(ne);
            const unsigned o = (unsigned)(cc.a[qq] - B);
            if (ne && o < (unsigned)P) atomicOr(&s_head[o / S], 1u << (o % S));
        });
        if (big)
            for (int rb = r0 + CR; rb <= stop;) {          // >= CR rows
                const int rq = min(rb + lane, stop);
                const int rp = row_ptr[rq];
                const unsigned o = (unsigned)(rp - B);
                const int rpn = row_ptr[rq + 1];
                const int vb = row_ptr[min(rb + kWave, stop + 1)];
                if (rb + kWave <= stop && read_lane(rp, 0) == vb) {
                    // 64 empty rows with more rows after them: skip the whole run
                    const int re = empty_run_end(row_ptr, rb + kWave, vb, stop);
                    lane_dirty = true;
                    zero_run(y, rb, re, lane);
                    rb = re;
                    continue;
                }
                if (rb + lane <= stop) {
                    if (rpn > rp) {
                        if (o < (unsigned)P) atomicOr(&s_head[o / S], 1u << (o % S));
                    } else {
                        lane_dirty = true;
                        y[rb + lane] = T(0);
                    }
                }
                rb += kWave;
            }
        dirty = ballot(lane_dirty) != 0ull;
        wave_sync();
        hb = s_head[lane];
        if (lane == 0) hb |= 1u;
        tile_transpose<T, S>(sb, prod, pc, lane);
        // ---- segment numbers
        const int nh = __popc(hb);
        const int incl = wave_incl_scan(nh, lane);
        seg_base = incl - nh;
        K = read_lane(incl, kWave - 1);
        partial_tail = (r1 < q.m) && (rp_r1 < B + P);
        // the tile loop starts a logical wave with a carry of +0
        if (lane == 0 && cont && wib == g0) pc[0] = pc[0] + T(0);
        acc = lane_segments(sb, pc, hb, seg_base, lane, T(0));
        present = ballot(hb != 0u);
        I = wave_segscan(acc, present, lane);
        out_val = read_lane(I, kWave - 1);
    } else {
        T s = prod[0];
#pragma unroll
        for (int k = 1; k < S; ++k) s += prod[k];
        s = wave_sum(s);
        out_val = (cont && wib == g0) ? T(0) + s : s;
    }

    bool lead_open = cont;       // the row open at the logical wave's start still is
    bool need = false;
    T carry = T(0);
    if (TPW > 1) {
        if (lane == 0) {
            sh.val[wib] = out_val;
            sh.kind[wib] = (general ? 0 : 1) | (cont ? 2 : 0);
        }
        __syncthreads();
        if (!active) return;
        if (wib > g0) {
            need = cont;
            const int kd = sh.kind[lane & (kMaxGroup - 1)];
            const unsigned fast = (unsigned)ballot(lane < kMaxGroup && (kd & 1));
            const unsigned conts = (unsigned)ballot(lane < kMaxGroup && (kd & 2));
            const unsigned below = ((1u << wib) - 1) & ~((1u << g0) - 1);   // its earlier tiles
            // the nearest earlier tile whose closing sum needs no carry
            const unsigned stops = below & ~(fast & conts);
            const int j = stops ? 31 - __builtin_clz(stops) : g0;
            carry = sh.val[j];
            for (int jj = j + 1; jj < wib; ++jj) carry = carry + sh.val[jj];
            lead_open = ((conts >> g0) & 1u) && (below & ~fast) == 0;
        }
    } else if (!active) {
        return;
    }
    const bool last = p == min((w + 1) * TPW, q.NP) - 1;
    [[maybe_unused]] const int wsh = __builtin_ctz(TPW * P);      // nonzero -> logical wave
    [[maybe_unused]] int sync_key = -1;
    [[maybe_unused]] T sync_v = T(0);
    if (general) {
        if (need) {
            // the carry starts lane 0's first sum: only the first segment changes
            T a0 = pc[0] + carry;
            unsigned hl = hb & ~1u;
#pragma unroll
            for (int kk = 1; kk < S; ++kk) {
                const T n = a0 + pc[kk];
                if (!(hl & ((2u << kk) - 1))) a0 = n;
            }
            if (lane == 0) {
                if (hl) sb[0] = a0;
                else acc = a0;
            }
            I = wave_segscan(acc, present, lane);
        }
        const T Iprev = dpp<kDppWaveShr1>(I);
        if (hb && lane > 0) sb[seg_base - 1] = Iprev + sb[seg_base - 1];
        if (lane == kWave - 1) sb[K - 1] = I;
        wave_sync();
        const int kb = lead_open ? 1 : 0;
        const int ke = partial_tail ? K - 1 : K;
        if (!dirty) {
            for (int kk = kb + lane; kk < ke; kk += kWave) y[(long long)r0 + kk] = alpha * sb[kk];
        } else {
            int running = 0;
            static_for<CP>([&](auto qc) {
                constexpr int qq = decltype(qc)::value;
                if (qq > 0 && r0 + qq * kWave > stop) return;
                const int row = r0 + qq * kWave + lane;
                const bool ne = __builtin_amdgcn_inverse_ballot_w64(mne[qq]);
                const int rank = running + popc_below(mne[qq]);
                if (ne && rank >= kb && rank < ke) y[row] = alpha * sb[rank];
                else if (row <= stop && !ne) y[row] = T(0);
                running += __popcll(mne[qq]);
            });
            if (big)
                for (int rb = r0 + CR; rb <= stop;) {
                    const int rq = min(rb + lane, stop);
                    const int rp = row_ptr[rq], rpn = row_ptr[rq + 1];
                    const int vb = row_ptr[min(rb + kWave, stop + 1)];
                    if (rb + kWave <= stop && read_lane(rp, 0) == vb) {
                        rb = empty_run_end(row_ptr, rb + kWave, vb, stop);   // no segments
                        continue;
                    }
                    const int r = rb + lane;
                    const bool ne = r <= stop && rpn > rp;
                    const uint64_t msk = ballot(ne);
                    const int rank = running + popc_below(msk);
                    if (ne && rank >= kb && rank < ke) y[r] = alpha * sb[rank];
                    running += __popcll(msk);
                    rb += kWave;
                }
        }
        if (lead_open) {     // the row began in an earlier logical wave and ends here
            if constexpr (FUSED)
                chain_add(cb, r0, read_lane(cc.a[0], 0) >> wsh, w, w, alpha * sb[0], lane, y);
            sync_key = r0;
            sync_v = alpha * sb[0];
        }
        if (last && partial_tail) {
            if constexpr (FUSED)
                chain_add(cb, r1, w, (rp_next - 1) >> wsh, w, alpha * sb[K - 1], lane, y);
            else if (lane == 0) y[r1] = alpha * sb[K - 1];
        }
    } else if (last) {
        const T tot = alpha * (need ? carry + out_val : out_val);
        if constexpr (FUSED) {
            const int first = lead_open ? read_lane(cc.a[0], 0) >> wsh : w;
            chain_add(cb, r1, first, (rp_next - 1) >> wsh, w, tot, lane, y);
        } else if (lead_open) {
            sync_key = r1;
            sync_v = tot;
        } else if (lane == 0) {
            y[r1] = tot;
        }
    }
    if constexpr (!FUSED) {
        // the wave that closes (or passes on) a row from an earlier logical
        // wave leaves its partial to calibrate_kernel; none: -1
        if (lane == 0 && (sync_key >= 0 || (wib == g0 && !cont))) {
            sync_row[w] = sync_key;
            if (sync_key >= 0) sync_val[w] = sync_v;
        }
    }
}

// ---------------------------------------------------------------------------
// Data-movement floor of a matrix: the main kernel's loads and gathers (same
// coalesced tile loads, same x gathers) with no segmentation and no y -- one
// wave per tile, one partial per lane.  Its time bounds what any CSR SpMV of
// the matrix can reach on the device.
// ---------------------------------------------------------------------------
template <typename T, int S>
__global__ __launch_bounds__(256) void floor_kernel(const int *__restrict__ col,
                                                   const T *__restrict__ val,
                                                   const T *__restrict__ x, int NP,
                                                   T *__restrict__ out)
{
    constexpr int P = kWave * S;
    const int lane = lane_id();
    const int p = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    if (p >= NP) return;
    Tile<T, S> t;
    tile_load<T, S>(col, val, p * P, lane, t);
    T xv[S];
#pragma unroll
    for (int k = 0; k < S; ++k) xv[k] = x[t.c[k]];
    T s = t.v[0] * xv[0];
#pragma unroll
    for (int k = 1; k < S; ++k) s += t.v[k] * xv[k];
    out[(long long)p * kWave + lane] = s;
}

// ---------------------------------------------------------------------------
// Calibration (bhsparse_spmv_cuda.h:166-173 moved to the device).  Every wave
// w wrote sync_row[w] (-1: none) and sync_val[w]; consecutive waves with the
// same row form a chain whose partials must be added, in wave order, to the
// value the row's starting wave stored.  One wave handles 64 consecutive
// entries: a segmented scan over runs of equal row gives each run's sum, the
// lane ending a run adds it to y; a run reaching past the window is extended
// window by window (wave sums).  Runs continuing from the previous window
// belong to the wave of that window.
// ---------------------------------------------------------------------------
// One window of 64 sync entries [base, base+64) for right-hand side rr.
// key(e) = sync_row[e] if entry e holds a partial of RHS rr, else -1.
template <typename T, int KMAX>
__device__ __forceinline__ void calibrate_window(const int *__restrict__ sync_row,
                                                 const T *__restrict__ sync_val,
                                                 const int *__restrict__ sync_k, int NW, int base,
                                                 int rr, int lane, T *__restrict__ y)
{
    auto key = [&](int e) -> int {
        if (e < 0 || e >= NW) return -1;
        const int r = sync_row[e];
        if (KMAX > 1 && r >= 0 && rr >= sync_k[e]) return -1;
        return r;
    };
    const int e = base + lane;
    const int r = key(e);
    const T v = r >= 0 ? sync_val[(long long)e * KMAX + rr] : T(0);
    const int before = key(base - 1);
    int rprev = dpp<kDppWaveShr1>(r);                 // lane i <- lane i-1
    if (lane == 0) rprev = before;
    const uint64_t starts = ballot(r != rprev) | 1ull;
    const T s = wave_segscan(v, starts, lane);
    const int rnext = dpp<kDppWaveShl1>(r);           // lane i <- lane i+1 (lane 63: unused)
    const bool run_end = (lane == kWave - 1) || (rnext != r);
    // the run holding lane 0 continues an earlier window's run?
    const int r0w = read_lane(r, 0);
    const bool lead_cont = r0w >= 0 && before == r0w;
    // run of lane 63 continuing into later windows
    const int r63 = read_lane(r, kWave - 1);
    T ext = T(0);
    if (r63 >= 0) {
        for (int nb = base + kWave; nb < NW; nb += kWave) {
            const int e2 = nb + lane;
            const int r2 = key(e2);
            const uint64_t same = ballot(r2 == r63);
            const int len = (same == ~0ull) ? kWave : __builtin_ctzll(~same);
            if (len == 0) break;
            const T v2 = lane < len ? sync_val[(long long)e2 * KMAX + rr] : T(0);
            ext = ext + wave_sum(v2);
            if (len < kWave) break;
        }
    }
    // lane's run starts at the last set bit of `starts` at or below it
    const uint64_t upto = starts & ((lane == 63) ? ~0ull : ((2ull << lane) - 1));
    const int run_start = 63 - __builtin_clzll(upto);
    const bool skip = (run_start == 0) && lead_cont;
    if (run_end && r >= 0 && !skip) {
        const T tot = (lane == kWave - 1) ? s + ext : s;
        y[(long long)r + rr] = y[(long long)r + rr] + tot;
    }
}

// ---------------------------------------------------------------------------
// Calibration (bhsparse_spmv_cuda.h:166-173 moved to the device).  Every wave
// w wrote sync_row[w] (-1: none) and sync_val[w]; consecutive waves with the
// same row form a chain whose partials must be added, in wave order, to the
// value the row's starting wave stored.  One wave handles 64 consecutive
// entries: a segmented scan over runs of equal row gives each run's sum, the
// lane ending a run adds it to y; a run reaching past the window is extended
// window by window (wave sums).  Runs continuing from the previous window
// belong to the wave of that window.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void calibrate_kernel(const int *__restrict__ sync_row,
                                                       const T *__restrict__ sync_val, int NW,
                                                       T *__restrict__ y)
{
    const int lane = lane_id();
    const int base = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6) * kWave;
    if (base >= NW) return;
    calibrate_window<T, 1>(sync_row, sync_val, nullptr, NW, base, 0, lane, y);
}

// ---------------------------------------------------------------------------
// Batched solves: many independent CSR matrices with up to KMAX right-hand
// sides each, in one persistent launch.  Every wave takes (matrix, wave-range)
// items from a global queue (one atomic per item) until the queue is empty --
// each wave exits once the counter passes n_items, so the grid always drains.
// The per-tile arithmetic is segsum_wave's, so a matrix/RHS pair gets exactly
// the bits a plain launch with the same tile shape gives.
// ---------------------------------------------------------------------------
struct BatchMeta {
    long long rp_off, tr_off, el_off, x_off, y_off;
    int sync_off, m, nnz, NP, NW, lead_empty, k, pad;
};

template <typename T, int S, int KMAX, int XCH>
__global__ __launch_bounds__(512) void batched_kernel(
    const int *__restrict__ row_ptr, const int *__restrict__ col, const T *__restrict__ val,
    const T *__restrict__ x, T *__restrict__ y, const int *__restrict__ tile_row,
    int *__restrict__ sync_row, T *__restrict__ sync_val, int *__restrict__ sync_k,
    const BatchMeta *__restrict__ meta, const int2 *__restrict__ items, int n_items,
    int *__restrict__ queue, int TPW, T alpha, int wave_lds_bytes)
{
    extern __shared__ double smem_raw[];
    const int lane = lane_id();
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    unsigned char *wave_lds = reinterpret_cast<unsigned char *>(smem_raw) + wib * wave_lds_bytes;
    unsigned *s_head = reinterpret_cast<unsigned *>(wave_lds);
    T *s_buf = reinterpret_cast<T *>(wave_lds + 256);   // room for 64*S pairs
    T *s_carry = s_buf + 2 * kWave * S;
    // XCH > 0: column indices and the x staging buffer after the carry
    unsigned char *s_stage =
        wave_lds + (256 + 2 * kWave * S * sizeof(T) + KMAX * sizeof(T) + 15) / 16 * 16;
    for (;;) {
        int it = 0;
        if (lane == 0) it = atomicAdd(queue, 1);
        it = __builtin_amdgcn_readfirstlane(it);
        if (it >= n_items) break;
        const int2 iw = items[it];
        const BatchMeta md = meta[iw.x];
        MatView<T> mv{row_ptr + md.rp_off, tile_row + md.tr_off, col + md.el_off,
                      val + md.el_off, x + md.x_off, y + md.y_off,
                      sync_row + md.sync_off, sync_val + (long long)md.sync_off * KMAX,
                      md.m, md.nnz, md.NP, md.NW, md.lead_empty, md.k, md.k, TPW,
                      (int)md.y_off};
        segsum_wave<T, S, KMAX, true, false, 2, XCH>(mv, iw.y, lane, s_head, s_buf,
                                                           s_carry, alpha, nullptr, s_stage);
        if (lane == 0) sync_k[md.sync_off + iw.y] = md.k;
        wave_sync();                              // LDS is reused by the next item
    }
}

// The same batch with one wave per tile (schedules of 1, 2, 4 or 8 tiles per
// wave without x staging): a block is one (matrix, logical wave) item, its waves
// the item's tiles, as in segsum_tiles_kernel.  The tile's stream, row boundaries
// and flags are read and made once; then the right-hand sides pass in pairs (k
// even, S * sizeof(T) <= 64 bytes; singly otherwise), the waves handing each
// pair's open partials over through LDS behind one barrier a pair.
//
// batched_kernel holds the tile after this one and the pair after this one in
// registers (176-256 VGPRs, 2 waves per SIMD, one right-hand side at a time
// where pairs do not fit) and starts few waves for small matrices; here pairs
// fit S = 8 in fp64 (156 VGPRs, 3 waves), and every tile has its wave at once.
// The kernel waits for x lines (k = 16: a 128-byte line per nonzero and pair).
// Replay of the graph, default schedule (S = 8, 4 tiles per wave), batched_kernel
// -> this: 24 matrices of 1,000-87,000 rows (10M nonzeros, 145M products) fp64
// 520 -> 249 us, fp32 341 -> 202; 24 of 1,000-4,000 rows 190 -> 47, 130 -> 42.
template <typename V>
struct BatchShare {
    V val[2][kMaxGroup];       // by parity of the pass: a wave may be one pass ahead
    int kind[kMaxGroup];       // bit 0: inside one row, bit 1: continues the row before it
};

template <typename T, int S, int KMAX>
__global__ __launch_bounds__(512) void batched_tiles_kernel(
    const int *__restrict__ row_ptr_all, const int *__restrict__ col_all,
    const T *__restrict__ val_all, const T *__restrict__ x_all, T *__restrict__ y_all,
    const int *__restrict__ tile_row_all, int *__restrict__ sync_row, T *__restrict__ sync_val,
    int *__restrict__ sync_k, const BatchMeta *__restrict__ meta, const int2 *__restrict__ items,
    int n_items, T alpha)
{
    constexpr int P = kWave * S, CP = 2, CR = CP * kWave;
    constexpr bool kPairs = S * sizeof(T) <= 64;
    using V2 = typename RhsVec<T, 2>::type;
    extern __shared__ double smem_raw[];
    const int lane = lane_id();
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int TPW = blockDim.x >> 6;
    // 16 neighbouring items per XCD (blocks are dealt round-robin over the 8):
    // they are mostly one matrix's neighbouring waves and share x lines in its L2
    constexpr int kRun = 16;
    int it = (int)blockIdx.x;
    if ((it / (8 * kRun) + 1) * (8 * kRun) <= n_items)
        it = it / (8 * kRun) * (8 * kRun) + (it % 8) * kRun + it / 8 % kRun;
    const int2 iw = items[it];
    const BatchMeta md = meta[iw.x];
    const int w = iw.y, p = w * TPW + wib;
    const int k = md.k;
    const int *__restrict__ row_ptr = row_ptr_all + md.rp_off;
    const int *__restrict__ tile_row = tile_row_all + md.tr_off;
    const T *__restrict__ x = x_all + md.x_off;
    T *__restrict__ y = y_all + md.y_off;
    constexpr int kBuf = P * (kPairs ? 2 : 1);
    T *s_buf = reinterpret_cast<T *>(smem_raw) + wib * kBuf;
    unsigned *s_head =
        reinterpret_cast<unsigned *>(reinterpret_cast<T *>(smem_raw) + TPW * kBuf) + wib * kWave;
    unsigned char *s_share = reinterpret_cast<unsigned char *>(
        reinterpret_cast<unsigned *>(reinterpret_cast<T *>(smem_raw) + TPW * kBuf) + TPW * kWave);
    const bool active = p < md.NP;
    const int pe = active ? p : 0;
    const int B = pe * P;

    Tile<T, S> t;
    tile_load<T, S>(col_all + md.el_off, val_all + md.el_off, B, lane, t);
    const int r0 = tile_row[pe], r1 = active ? tile_row[pe + 1] : r0;
    const RowChunk<CP> cc = load_chunk<CP>(row_ptr, r0, lane, md.m);
    const int rp_r1 = row_ptr[min(r1, md.m)];
    if (md.lead_empty > 0 && active) {
        const unsigned n = (unsigned)md.lead_empty * k;      // a batch's y is below 2^31
        const unsigned per = (n + (unsigned)md.NP - 1) / (unsigned)md.NP, lo = (unsigned)p * per;
        for (unsigned r = lo + lane; r < lo + per && r < n; r += kWave) y[r] = T(0);
    }
    const bool tail = B + P > md.nnz;
    const bool general = r0 != r1;
    const bool cont = read_lane(cc.a[0], 0) < B;
    const int stop = (r1 == md.m) ? md.m - 1 : r1;
    const bool big = r1 - r0 >= CR;
    uint64_t mne[CP];
    unsigned hb = 0;
    bool dirty = false, partial_tail = false;
    int seg_base = 0, K = 0;
    uint64_t present = 1;
    if (general) {
        bool lane_dirty = false;
        s_head[lane] = 0u;
        wave_sync();
        static_for<CP>([&](auto qc) {
            constexpr int qq = decltype(qc)::value;
            mne[qq] = 0ull;
            if (qq > 0 && r0 + qq * kWave > stop) return;   // wave-uniform: no rows here
            const bool have = r0 + qq * kWave + lane <= stop;
            const bool ne = have && chunk_next<qq>(cc, lane) > cc.a[qq];
            lane_dirty = lane_dirty || (have && !ne);
            mne[qq] = ballot(ne);
            const unsigned o = (unsigned)(cc.a[qq] - B);
            if (ne && o < (unsigned)P) atomicOr(&s_head[o / S], 1u << (o % S));
        });
        if (big)
            for (int rb = r0 + CR; rb <= stop;) {          // >= CR rows
                const int rq = min(rb + lane, stop);
                const int rp = row_ptr[rq], rpn = row_ptr[rq + 1];
                const int vb = row_ptr[min(rb + kWave, stop + 1)];
                if (rb + kWave <= stop && read_lane(rp, 0) == vb) {
                    // 64 empty rows with more rows after them: skip the whole run
                    const int re = empty_run_end(row_ptr, rb + kWave, vb, stop);
                    lane_dirty = true;
                    zero_run(y, (long long)rb * k, (long long)re * k, lane);
                    rb = re;
                    continue;
                }
                if (rb + lane <= stop) {
                    const unsigned o = (unsigned)(rp - B);
                    if (rpn > rp) {
                        if (o < (unsigned)P) atomicOr(&s_head[o / S], 1u << (o % S));
                    } else {
                        lane_dirty = true;
                        for (int rr = 0; rr < k; ++rr) y[(long long)(rb + lane) * k + rr] = T(0);
                    }
                }
                rb += kWave;
            }
        dirty = ballot(lane_dirty) != 0ull;
        wave_sync();
        hb = s_head[lane];
        if (lane == 0) hb |= 1u;
        const int nh = __popc(hb);
        const int incl = wave_incl_scan(nh, lane);
        seg_base = incl - nh;
        K = read_lane(incl, kWave - 1);
        partial_tail = (r1 < md.m) && (rp_r1 < B + P);
        present = ballot(hb != 0u);
    }
    const bool last = p == min((w + 1) * TPW, md.NP) - 1;
    bool lead_open = cont;       // the row open at the item's start still is
    int from = 0;                // the nearest earlier tile whose closing sum needs no carry

    auto pass = [&](auto rt, int rr, int turn) __attribute__((always_inline)) {
        constexpr int R = decltype(rt)::value;
        using V = typename RhsVec<T, R>::type;
        const V zero = static_cast<V>(T(0));
        V *sb = reinterpret_cast<V *>(s_buf);
        BatchShare<V> &sh = *reinterpret_cast<BatchShare<V> *>(s_share);
        V acc = zero, I = zero, out_val, pc[S];
        {
            V prod[S];
#pragma unroll
            for (int kk = 0; kk < S; ++kk)
                prod[kk] = *reinterpret_cast<const V *>(x + (long long)t.c[kk] * k + rr);
#pragma unroll
            for (int kk = 0; kk < S; ++kk) prod[kk] = t.v[kk] * prod[kk];
            if (tail) {
#pragma unroll
                for (int kk = 0; kk < S; ++kk)
                    prod[kk] = keep_or_zero(prod[kk], tile_item<T, S>(B, lane, kk) < md.nnz);
            }
            if (general) {
                wave_sync();                 // the pass before has read its segments
                tile_transpose<T, S>(sb, prod, pc, lane);
                // the tile loop starts a logical wave with a carry of +0
                if (lane == 0 && cont && wib == 0) pc[0] = pc[0] + zero;
                acc = lane_segments(sb, pc, hb, seg_base, lane, zero);
                I = wave_segscan(acc, present, lane);
                out_val = read_lane(I, kWave - 1);
            } else {
                V s = prod[0];
#pragma unroll
                for (int kk = 1; kk < S; ++kk) s += prod[kk];
                s = wave_sum(s);
                out_val = (cont && wib == 0) ? zero + s : s;
            }
        }
        V carry = zero;
        const bool need = cont && wib > 0;
        if (TPW > 1) {
            if (lane == 0) {
                sh.val[turn & 1][wib] = out_val;
                if (turn == 0) sh.kind[wib] = (general ? 0 : 1) | (cont ? 2 : 0);
            }
            __syncthreads();
            if (wib > 0) {
                if (turn == 0) {
                    const int kd = sh.kind[lane & (kMaxGroup - 1)];
                    const unsigned fast = (unsigned)ballot(lane < kMaxGroup && (kd & 1));
                    const unsigned conts = (unsigned)ballot(lane < kMaxGroup && (kd & 2));
                    const unsigned below = (1u << wib) - 1;
                    const unsigned stops = below & ~(fast & conts);
                    from = stops ? 31 - __builtin_clz(stops) : 0;
                    lead_open = (conts & 1u) && (below & ~fast) == 0;
                }
                carry = sh.val[turn & 1][from];
                for (int j = from + 1; j < wib; ++j) carry = carry + sh.val[turn & 1][j];
            }
        }
        if (!active) return;
        auto store_y = [&](long long row, V v) {
            *reinterpret_cast<V *>(y + row * k + rr) = v;
        };
        V *sv = reinterpret_cast<V *>(sync_val + (long long)(md.sync_off + w) * KMAX + rr);
        if (general) {
            if (need) {
                // the carry starts lane 0's first sum: only the first segment changes
                V a0 = pc[0] + carry;
                const unsigned hl = hb & ~1u;
#pragma unroll
                for (int kk = 1; kk < S; ++kk) {
                    const V n = a0 + pc[kk];
                    if (!(hl & ((2u << kk) - 1))) a0 = n;
                }
                if (lane == 0) {
                    if (hl) sb[0] = a0;
                    else acc = a0;
                }
                I = wave_segscan(acc, present, lane);
            }
            const V Iprev = dpp<kDppWaveShr1>(I);
            if (hb && lane > 0) sb[seg_base - 1] = Iprev + sb[seg_base - 1];
            if (lane == kWave - 1) sb[K - 1] = I;
            wave_sync();
            const int kb = lead_open ? 1 : 0;
            const int ke = partial_tail ? K - 1 : K;
            if (!dirty) {
                for (int kk = kb + lane; kk < ke; kk += kWave) store_y(r0 + kk, alpha * sb[kk]);
            } else {
                int running = 0;
                static_for<CP>([&](auto qc) {
                    constexpr int qq = decltype(qc)::value;
                    if (qq > 0 && r0 + qq * kWave > stop) return;
                    const int row = r0 + qq * kWave + lane;
                    const bool ne = __builtin_amdgcn_inverse_ballot_w64(mne[qq]);
                    const int rank = running + popc_below(mne[qq]);
                    if (ne && rank >= kb && rank < ke) store_y(row, alpha * sb[rank]);
                    else if (row <= stop && !ne) store_y(row, zero);
                    running += __popcll(mne[qq]);
                });
                if (big)
                    for (int rb = r0 + CR; rb <= stop;) {
                        const int rq = min(rb + lane, stop);
                        const int rp = row_ptr[rq], rpn = row_ptr[rq + 1];
                        const int vb = row_ptr[min(rb + kWave, stop + 1)];
                        if (rb + kWave <= stop && read_lane(rp, 0) == vb) {
                            rb = empty_run_end(row_ptr, rb + kWave, vb, stop);   // no segments
                            continue;
                        }
                        const int r = rb + lane;
                        const bool ne = r <= stop && rpn > rp;
                        const uint64_t msk = ballot(ne);
                        const int rank = running + popc_below(msk);
                        if (ne && rank >= kb && rank < ke) store_y(r, alpha * sb[rank]);
                        running += __popcll(msk);
                        rb += kWave;
                    }
            }
            if (lane == 0) {
                if (lead_open) *sv = alpha * sb[0];
                if (last && partial_tail) store_y(r1, alpha * sb[K - 1]);
            }
        } else if (last && lane == 0) {
            const V tot = alpha * (need ? carry + out_val : out_val);
            if (lead_open) *sv = tot;
            else store_y(r1, tot);
        }
    };
    bool done = false;
    if constexpr (kPairs) {
        if ((k & 1) == 0) {
            for (int rr = 0; rr < k; rr += 2) pass(RhsTag<2>{}, rr, rr >> 1);
            done = true;
        }
    }
    if (!done)
        for (int rr = 0; rr < k; ++rr) pass(RhsTag<1>{}, rr, rr);
    // the wave that closes (or passes on) a row from an earlier item says which
    if (active && lane == 0) {
        const bool sent = lead_open && (general || last);
        if (sent || (wib == 0 && !cont)) {
            sync_row[md.sync_off + w] = sent ? (int)md.y_off + (general ? r0 : r1) * k : -1;
            sync_k[md.sync_off + w] = k;
        }
    }
}

// Calibration of a batch: sync entries of each matrix start on a multiple of
// 64, so every window lies inside one matrix and matches the windows of that
// matrix's own plain calibration; keys are y slots (unique across the batch).
template <typename T, int KMAX>
__global__ __launch_bounds__(256) void calibrate_batched_kernel(const int *__restrict__ sync_row,
                                                               const T *__restrict__ sync_val,
                                                               const int *__restrict__ sync_k,
                                                               int NW, T *__restrict__ y)
{
    const int lane = lane_id();
    const int base = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6) * kWave;
    if (base >= NW) return;
    const int rr = (int)blockIdx.y;                // one right-hand side per grid row
    const int e = base + lane;
    if (ballot(e < NW && sync_row[e] >= 0 && sync_k[e] > rr) == 0ull) return;
    calibrate_window<T, KMAX>(sync_row, sync_val, sync_k, NW, base, rr, lane, y);
}

// y[i] = sum over panels p (in order) of row i's panel partial, +0 where row i
// has no entry in panel p.  The last step of the column-panel variant; every
// partial already carries alpha.  A wave covers GROUPS groups of 64 rows; for
// group g, bit p of mask[i] says row i has entries in panel p, and that
// partial is stacked row base[g*NPAN+p] + (rows of the group below i with bit
// p set), a ballot and a popcount.  Reads m bytes of mask instead of an
// NPAN x m index map.  All partials of the wave's rows are loaded before any
// is added, so each wave has GROUPS*NPAN loads in flight.
//
// The calibration of the stacked matrix is done here too (no calibrate_kernel
// launch on this layout).  A stacked row whose nonzeros cross wave boundaries
// has a chain of consecutive waves that each left a partial in sync_val; the
// chains depend only on the stacked matrix and the tile shape, so they are
// listed once per analysis as ChainRec records: combine wave cw has
// kChainSlots slots chains[cw * kChainSlots + j] (count 0: empty), filled in
// order, and the last slot's `next` links any further records.  The slots are
// loaded with the masks, and the first 64 partials of every slot's chain with
// the panel partials, so that a combine wave's chains add no round trip to
// memory unless it has more than kChainSlots of them or one of more than 64
// waves.  A chain's total is summed 64 entries at a time (wave_sum of each
// chunk, the chunk sums in order) and added to that partial before the panel
// sum: y_stack[R] + total, the value calibrate_kernel would have stored.  A
// stacked row has at most one chain, so chains never meet in one partial.
struct ChainRec {
    int first;   // first wave of the chain (its sync_val index)
    int count;   // waves in the chain (0: no record)
    int where;   // (row - first row of the combine wave) << 4 | panel
    int next;    // index of the next record of the same combine wave, -1: none
};
constexpr int kCombineGroups = 2;   // 64-row groups per combine wave
constexpr int kChainSlots = 4;      // chain records per combine wave loaded up front

template <typename T, int NPAN, int GROUPS>
__global__ __launch_bounds__(256) void combine_panels_kernel(const T *__restrict__ ystack,
                                                            const unsigned char *__restrict__ mask,
                                                            const int *__restrict__ base, int m,
                                                            T *__restrict__ y,
                                                            const ChainRec *__restrict__ chains,
                                                            const T *__restrict__ sync_val)
{
    const int lane = lane_id();
    const int cw = __builtin_amdgcn_readfirstlane(
        (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const long long g0 = (long long)cw * GROUPS;
    if (g0 * kWave >= m) return;                      // whole wave past the last row
    // chain slots, masks and bases first, so that no wait for them also waits
    // for partials already in flight
    ChainRec slot{0, 0, 0, -1};
    if (lane < kChainSlots) slot = chains[(long long)cw * kChainSlots + lane];
    unsigned mk[GROUPS];
    int gb[GROUPS][NPAN];
#pragma unroll
    for (int h = 0; h < GROUPS; ++h) {
        const long long g = g0 + h;
        const long long i = g * kWave + lane;
        mk[h] = i < m ? (unsigned)mask[i] : 0u;          // no bits past the last row
        const int *b = base + (g * kWave < m ? g : g0) * NPAN;
#pragma unroll
        for (int p = 0; p < NPAN; ++p) gb[h][p] = b[p];
    }
    T v[GROUPS][NPAN];
#pragma unroll
    for (int h = 0; h < GROUPS; ++h) {
#pragma unroll
        for (int p = 0; p < NPAN; ++p) {
            const bool has = (mk[h] >> p) & 1u;
            const uint64_t bits = ballot(has);         // every lane of the wave is active
            const int pos = has ? gb[h][p] + popc_below(bits) : 0;
            v[h][p] = has ? ystack[pos] : T(0);
        }
    }
    // the first chunk of every slot's chain, in flight with the partials
    int c_first[kChainSlots], c_count[kChainSlots], c_where[kChainSlots];
    T c0[kChainSlots];
#pragma unroll
    for (int j = 0; j < kChainSlots; ++j) {
        c_first[j] = read_lane(slot.first, j);
        c_count[j] = read_lane(slot.count, j);
        c_where[j] = read_lane(slot.where, j);
        c0[j] = lane < c_count[j] ? sync_val[(long long)c_first[j] + lane] : T(0);
    }
    auto add_chain = [&](int first, int count, int where, T s) {
        T tot = wave_sum(s);
        for (int j = kWave; j < count; j += kWave)
            tot = tot + wave_sum(j + lane < count ? sync_val[(long long)first + j + lane] : T(0));
        const int row = where >> 4, pan = where & 15;
#pragma unroll
        for (int h = 0; h < GROUPS; ++h)
#pragma unroll
            for (int p = 0; p < NPAN; ++p)
                if (pan == p && row == h * kWave + lane) v[h][p] = v[h][p] + tot;
    };
#pragma unroll
    for (int j = 0; j < kChainSlots; ++j)
        if (c_count[j] > 0) add_chain(c_first[j], c_count[j], c_where[j], c0[j]);
    for (int nx = read_lane(slot.next, kChainSlots - 1); nx >= 0;) {   // wave-uniform
        const ChainRec c = chains[nx];
        add_chain(c.first, c.count, c.where,
                  lane < c.count ? sync_val[(long long)c.first + lane] : T(0));
        nx = c.next;
    }
#pragma unroll
    for (int h = 0; h < GROUPS; ++h) {
        const long long i = (g0 + h) * kWave + lane;
        T s = v[h][0];
#pragma unroll
        for (int p = 1; p < NPAN; ++p) s += v[h][p];    // panel order
        if (i < m) y[i] = s;
    }
}

// ---------------------------------------------------------------------------
// Device build of the column-panel copy (count -> scan -> scatter).  Panel of
// column c: c / pw.  The stacked matrix has one row per nonempty (panel, row)
// pair, panel-major; within a stacked row the entries keep their order in A.
// ---------------------------------------------------------------------------
// cnt[p*m + i] = entries of row i in panel p; mask[i] bit p = (cnt > 0).  One
// wave per row, 64 entries at a time (a row may hold 10^5 entries).
template <int NPAN>
__global__ __launch_bounds__(256) void panel_count_kernel(const int *__restrict__ row_ptr,
                                                         const int *__restrict__ col, int m,
                                                         int pw, int *__restrict__ cnt,
                                                         unsigned char *__restrict__ mask)
{
    const int lane = lane_id();
    const long long i = __builtin_amdgcn_readfirstlane(
        (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    if (i >= m) return;
    const int b = row_ptr[i], e = row_ptr[i + 1];
    int c[NPAN];
#pragma unroll
    for (int p = 0; p < NPAN; ++p) c[p] = 0;
    for (int j = b; j < e; j += kWave) {
        const int q = j + lane < e ? col[j + lane] / pw : -1;
#pragma unroll
        for (int p = 0; p < NPAN; ++p) c[p] += __popcll(ballot(q == p));
    }
    if (lane == 0) {
        unsigned mk = 0;
#pragma unroll
        for (int p = 0; p < NPAN; ++p) {
            cnt[(long long)p * m + i] = c[p];
            mk |= (c[p] > 0 ? 1u : 0u) << p;
        }
        mask[i] = (unsigned char)mk;
    }
}

// With flag[q] = (cnt[q] > 0) and rows[q] / nzs[q] the exclusive sums of the
// flags / counts over q = p*m + i: the stacked row of a nonempty pair is
// rows[q]; its start is nzs[q]; base[g*NPAN + p] = rows[p*m + 64g] is the first
// stacked row of panel p at or after row 64g (read only for groups that have
// rows in panel p); owner[R] = the row of A that stacked row R belongs to.
template <int NPAN>
__global__ __launch_bounds__(256) void panel_index_kernel(const int *__restrict__ cnt,
                                                         const int *__restrict__ rows,
                                                         const int *__restrict__ nzs, int m,
                                                         int *__restrict__ prow_ptr,
                                                         int *__restrict__ owner,
                                                         int *__restrict__ base)
{
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)NPAN * m) return;
    const int p = (int)(q / m), i = (int)(q % m);
    if (cnt[q] > 0) {
        prow_ptr[rows[q]] = nzs[q];
        owner[rows[q]] = i;
    }
    if ((i & 63) == 0) base[(long long)(i >> 6) * NPAN + p] = rows[q];
}

// Entries of row i to their stacked rows, in order: one wave per row, 64
// entries at a time; an entry's place is its panel's running offset plus the
// number of lower lanes in the same panel (ballot + mbcnt).
template <typename T, int NPAN>
__global__ __launch_bounds__(256) void panel_scatter_kernel(
    const int *__restrict__ row_ptr, const int *__restrict__ col, const T *__restrict__ val,
    int m, int pw, const int *__restrict__ cnt, const int *__restrict__ nzs,
    int *__restrict__ pcol, T *__restrict__ pval)
{
    const int lane = lane_id();
    const long long i = __builtin_amdgcn_readfirstlane(
        (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    if (i >= m) return;
    const int b = row_ptr[i], e = row_ptr[i + 1];
    int off[NPAN];
#pragma unroll
    for (int p = 0; p < NPAN; ++p) off[p] = nzs[(long long)p * m + i];
    for (int j = b; j < e; j += kWave) {
        const bool in = j + lane < e;
        const int c = in ? col[j + lane] : 0;
        const T v = in ? val[j + lane] : T(0);
        const int q = in ? c / pw : -1;
        int d = 0;
#pragma unroll
        for (int p = 0; p < NPAN; ++p) {
            const uint64_t bits = ballot(q == p);
            if (q == p) d = off[p] + popc_below(bits);
            off[p] += __popcll(bits);
        }
        if (in) {
            pcol[d] = c;
            pval[d] = v;
        }
    }
}

// Copies `words` 32-bit words in pieces of kPieceBytes, one end of the copy pinned
// host memory, and sets flags[p * flag_step] = tag behind piece p: to the host, when
// its data are there; from the host, when they have been read (what follows on the
// stream finds them; a release to the system here would write the L2 back, 15 us).
// Blocks take the pieces in turn, so they are done in about their order.  src
// and dst on 16 bytes; a launch moves 2 MB at most, so 32-bit sizes do.
constexpr int kPieceBytes = 16384;

template <bool TO_HOST>
__global__ __launch_bounds__(256) void copy_pieces_kernel(const unsigned *__restrict__ src,
                                                          unsigned *__restrict__ dst, int words,
                                                          unsigned *flags, int flag_step,
                                                          unsigned tag)
{
    constexpr int W = kPieceBytes / 4;
    for (int p = blockIdx.x; p * W < words; p += gridDim.x) {
        const unsigned *s = src + p * W;
        unsigned *d = dst + p * W;
        const int n = min(words - p * W, W);
        u32x4 v[W / 1024];                // all of a thread's loads on their way at once
#pragma unroll
        for (int i = 0; i < W / 1024; ++i) {
            const int at = i * 256 + (int)threadIdx.x;
            if (at < n / 4) v[i] = reinterpret_cast<const u32x4 *>(s)[at];
        }
#pragma unroll
        for (int i = 0; i < W / 1024; ++i) {
            const int at = i * 256 + (int)threadIdx.x;
            if (at < n / 4) reinterpret_cast<u32x4 *>(d)[at] = v[i];
        }
        if ((int)threadIdx.x < n % 4) d[n / 4 * 4 + threadIdx.x] = s[n / 4 * 4 + threadIdx.x];
        if constexpr (TO_HOST) __threadfence_system();
        __syncthreads();                  // every wave's data are there, or read
        if (threadIdx.x == 0)
            __hip_atomic_store(flags + p * flag_step, tag, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Tells the host that the stream has come here.
__global__ void signal_kernel(unsigned *flag, unsigned tag)
{
    __hip_atomic_store(flag, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Whether row_ptr is monotone (else *bad |= 1) and every column index lies in
// [0, n) (else *bad |= 2): one read of row_ptr and col, col in 16-byte loads
// (both from hipMalloc).
__global__ __launch_bounds__(256) void check_csr_kernel(const int *__restrict__ row_ptr,
                                                        const int *__restrict__ col, int m, int n,
                                                        int nnz, int *__restrict__ bad)
{
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x, step = (long long)gridDim.x * 256;
    int b = 0;
    for (long long i = t; i < m; i += step) b |= row_ptr[i + 1] < row_ptr[i];
    const u32x4 *c4 = reinterpret_cast<const u32x4 *>(col);
    const unsigned un = (unsigned)n;
    for (long long i = t; i < nnz / 4; i += step) {
        const u32x4 c = c4[i];
        if (c.x >= un || c.y >= un || c.z >= un || c.w >= un) b |= 2;
    }
    if (t < nnz % 4 && (unsigned)col[nnz - 1 - t] >= un) b |= 2;
    if (b) atomicOr(bad, b);
}

// The right-hand sides of a batch one after another, for its per-vector
// launches: xp[off + r * n + j] = x[off + j * k + r].  `per_mat` blocks a matrix;
// a thread moves a column's k values, consecutive in x, and a wave's stores are
// consecutive for each r.
struct BatchX {
    long long off;
    int n, k;
};

template <typename T>
__global__ __launch_bounds__(256) void rhs_major_kernel(const T *__restrict__ x, T *__restrict__ xp,
                                                        const BatchX *__restrict__ bx, int n_mats,
                                                        int per_mat)
{
    for (long long i = blockIdx.x / per_mat; i < n_mats; i += gridDim.x / per_mat) {
        const BatchX b = bx[i];
        for (long long j = (long long)(blockIdx.x % per_mat) * 256 + threadIdx.x; j < b.n;
             j += (long long)per_mat * 256)
            for (int r = 0; r < b.k; ++r)
                xp[b.off + (long long)r * b.n + j] = x[b.off + j * b.k + r];
    }
}

template <typename T>
__global__ __launch_bounds__(256) void fill_kernel(T *__restrict__ p, long long n, T v)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

// Writes `n16` 16-byte words; used to push earlier data out of L2 and MALL.
__global__ __launch_bounds__(256) void flush_kernel(u32x4 *__restrict__ p, long long n16, unsigned v)
{
    const u32x4 z = {v, v, v, v};
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n16;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = z;
}

// Plain copy of n16 16-byte words (bandwidth probe and counter calibration).
__global__ __launch_bounds__(256) void copy_kernel(const u32x4 *__restrict__ src,
                                                  u32x4 *__restrict__ dst, long long n16)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n16;
         i += (long long)gridDim.x * blockDim.x)
        dst[i] = __builtin_nontemporal_load(src + i);
}

// ---------------------------------------------------------------------------
// csr-vector (kernels_cuda.h:272-342, CUSP v0.4.0; wave64 form of
// csr_vector_spmv_kernels.cl:10-78): TPV lanes per row, lane-strided partial
// sums, then a shuffle tree replacing the LDS tree; rows longer than 64 with
// TPV = 64 start at an aligned index (:307-320).
// ---------------------------------------------------------------------------
template <typename T, int TPV>
__global__ __launch_bounds__(256) void csrvec_kernel(int m, const int *__restrict__ row_ptr,
                                                    const int *__restrict__ col,
                                                    const T *__restrict__ val,
                                                    const T *__restrict__ x, T *__restrict__ y,
                                                    T alpha, long long x_lines)
{
    const int tl = threadIdx.x & (TPV - 1);
    const long long vid = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / TPV;
    const long long nv = (long long)gridDim.x * blockDim.x / TPV;
    // x_lines > 0 (x small enough for every L2): the blocks of each XCD (dealt
    // round-robin, block b on XCD b % 8) read one word of every 128-byte line
    // of x between them, so x is on its way into that XCD's L2 while row_ptr
    // and the entries are loaded, and the gathers after them hit it.
    int touch = 0;
    {
        const long long t = (long long)(blockIdx.x / 8) * blockDim.x + threadIdx.x;
        if (t < x_lines) touch = reinterpret_cast<const int *>(x)[t * (128 / sizeof(int))];
    }
    for (long long row = vid; row < m; row += nv) {
        const int rs = row_ptr[row], re = row_ptr[row + 1];
        T sum = T(0);
        if (TPV == kWave && re - rs > kWave) {
            int jj = rs - (rs & (TPV - 1)) + tl;
            if (jj >= rs && jj < re) sum += val[jj] * x[col[jj]];
            for (jj += TPV; jj < re; jj += TPV) sum += val[jj] * x[col[jj]];
        } else {
            for (int jj = rs + tl; jj < re; jj += TPV) sum += val[jj] * x[col[jj]];
        }
#pragma unroll
        for (int off = TPV / 2; off > 0; off >>= 1) sum += __shfl_down(sum, off, TPV);
        if (tl == 0) y[row] = alpha * sum;
    }
    asm volatile("" ::"v"(touch));   // keeps the touch load; emits no instruction
}

// ---------------------------------------------------------------------------
// Row-length statistics for the tuner: sums of len and len^2, max len, empty
// rows and the summed column span (last - first + 1) of nonempty rows, as
// exact 64-bit integers (one atomic per block).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void row_stats_kernel(int m, const int *__restrict__ row_ptr,
                                                       const int *__restrict__ col,
                                                       unsigned long long *__restrict__ out)
{
    unsigned long long s1 = 0, s2 = 0, se = 0, ssp = 0;
    unsigned mx = 0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < m;
         i += (long long)gridDim.x * blockDim.x) {
        const int b = row_ptr[i], e = row_ptr[i + 1];
        const unsigned L = (unsigned)(e - b);
        s1 += L;
        s2 += (unsigned long long)L * L;
        mx = L > mx ? L : mx;
        if (L == 0) se++;
        else ssp += (unsigned long long)(col[e - 1] - col[b] + 1);
    }
    __shared__ unsigned long long red[4][4];
    __shared__ unsigned redm[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s1 += __shfl_xor(s1, off, kWave);
        s2 += __shfl_xor(s2, off, kWave);
        se += __shfl_xor(se, off, kWave);
        ssp += __shfl_xor(ssp, off, kWave);
        unsigned o = __shfl_xor(mx, off, kWave);
        mx = o > mx ? o : mx;
    }
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[wv][0] = s1; red[wv][1] = s2; red[wv][2] = se; red[wv][3] = ssp;
        redm[wv] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = blockDim.x >> 6;
        for (int i = 1; i < nw; ++i) {
            s1 += red[i][0]; s2 += red[i][1]; se += red[i][2]; ssp += red[i][3];
            mx = redm[i] > mx ? redm[i] : mx;
        }
        atomicAdd(&out[0], s1);
        atomicAdd(&out[1], s2);
        atomicAdd(&out[2], se);
        atomicAdd(&out[3], ssp);
        atomicMax(&out[4], (unsigned long long)mx);
    }
}

} // namespace bhs
