// kernels.hip -- HIP kernels of the HSMU SpGEMM path for gfx950 (MI355X).
//
// Pipeline for C = A * B (all on one stream; host synchronises twice, to validate the
// input / size the symbolic launches and to size C):
//   1. B -> 64-column tiles (k_btiles: one pass, chained scan; for a B of short rows only
//      the rows' records, k_brows, unless a row of C wants the tiles).
//      Reference: src/compressed/compressed_mask64.cuh:61-424.  Tiles of a row come out
//      sorted by tile column (the reference's order is whatever LDS atomics give).
//   2. Row analysis of A (k_row_info): products, tile-products and the tile span
//      [rmin, rmax] of each row of C.  Reference: k_compute_flop, src/small/mask.cuh:14-51.
//   3. Binning (in k_row_info, and in k_rowptr_bin for the numeric phase) by work and LDS
//      need, wave/workgroup-aggregated appends.  Reference: src/bining.cuh:1-395 (fixed
//      ranges there; derived from LDS need here).
//   4. Symbolic (k_symbolic_row / _wide / _global): OR of B's tile masks over the A row
//      into a mask directory over the row's tile span, nnz(C_i) = sum popcount; rows of few
//      products (k_small_bin, k_small_rows) mark their columns directly.
//      Reference: compressed_tilePtr_symbolic.cuh + compressed_tileOR.cuh, which do the
//      same in two hash passes; the dense directory needs one pass and no hashing.
//   5. Scan of nnz(C_i) to row pointers (k_rowptr_bin).
//   6. Numeric (k_numeric_row, k_small_bin, k_numeric_windows): the HSMU accumulator.  The row's
//      value array is exactly nnz(C_i) long; the slot of column c is
//        off[t] + popcount(mask[t] & ((1 << (c & 63)) - 1)),  t = (c >> 6) - rmin,
//      i.e. the rank of c among C's sorted columns, found in O(1) from the tile
//      directory where the reference binary-searches a sorted column list
//      (src/compressed/compressed_Cval.cuh:5-69, src/small/numeric.cuh:233-253).
//      The same kernel writes C's sorted columns by expanding the tile masks, which
//      replaces the reference's separate O(n^2) rank-sort pass
//      (src/compressed/compressed_Ccol_symbolic.cuh:4-63).
//   Rows whose directory + values do not fit LDS: the symbolic tile OR runs on a global
//   workspace, the numeric phase takes the row in windows of its columns (the reference's
//   bin-13 dense spECK path, src/external/spECK/dense_acc.cu:246-267, whose early return
//   leaves rows unwritten; every row is written here).

#include <hip/hip_runtime.h>

#include <climits>

#include "device_common.h"
#include "hsmu_internal.h"

namespace hsmu {

// ---- fill / copy -------------------------------------------------------------------

__global__ __launch_bounds__(256) void k_fill_zero(uint4 *p, size_t n16, unsigned char *tail, size_t ntail)
{
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += stride)
        p[i] = make_uint4(0, 0, 0, 0);
    if (blockIdx.x == 0 && threadIdx.x < ntail)
        tail[threadIdx.x] = 0;
}

hipError_t launch_fill_zero(void *p, size_t bytes, hipStream_t s)
{
    if (bytes == 0)
        return hipSuccess;
    const size_t n16 = bytes / 16;
    const size_t ntail = bytes - n16 * 16;
    size_t blocks = (n16 + 255) / 256;
    if (blocks > 4096)
        blocks = 4096;
    if (blocks == 0)
        blocks = 1;
    hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)blocks), dim3(256), 0, s, (uint4 *)p, n16,
                       (unsigned char *)p + n16 * 16, ntail);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16)
{
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += stride)
        dst[i] = src[i];
}

hipError_t launch_copy(const void *src, void *dst, size_t bytes, int num_cus, hipStream_t s)
{
    const size_t n16 = bytes / 16;
    size_t blocks = (n16 + 255) / 256;
    const size_t cap = (size_t)num_cus * 16;
    if (blocks > cap)
        blocks = cap;
    if (blocks == 0)
        blocks = 1;
    hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, s, (const uint4 *)src, (uint4 *)dst, n16);
    return hipGetLastError();
}

// Loads and stores at the device's point of coherence, beside the atomics' updates.
template <typename T> DEVI T device_load(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> DEVI void device_store(T *p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- chained scan ---------------------------------------------------------------------
//
// Blocks take their place in a sequence from a counter (so that a block only ever waits for
// blocks that are running), publish the sum of their part and then the prefix up to their
// end, and read back over their predecessors' words until one holds a prefix.  A word holds
// its state and its value together, so no other memory has to be ordered.
constexpr u64 CHAIN_SUM = 1ull << 62, CHAIN_PREFIX = 2ull << 62, CHAIN_VALUE = CHAIN_SUM - 1;

// The sum of the parts before place `b`; `part` is this block's.  Called by one whole wave.
DEVI u64 chain_prefix(u64 *words, int b, u64 part)
{
    const int lane = threadIdx.x & 63;
    if (lane == 0)
        device_store(&words[b], (b ? CHAIN_SUM : CHAIN_PREFIX) | part);
    // CHAIN_W words per lane at a time: blocks of one launch publish together, so most find
    // sums only, all the way back, and every round costs a trip to memory
    constexpr int CHAIN_W = 4;
    u64 before = 0;
    for (int e = b; e > 0;) { // words [e - 64 CHAIN_W, e), the nearest first
        u64 w[CHAIN_W];
#pragma unroll
        for (int i = 0; i < CHAIN_W; ++i) {
            const int q = e - 1 - lane - 64 * i;
            w[i] = q >= 0 ? device_load(&words[q]) : CHAIN_PREFIX; // before the first: a prefix of 0
        }
        bool wait = false, found = false;
        u64 sum = 0;
        int used = 0;
#pragma unroll
        for (int i = 0; i < CHAIN_W; ++i) {
            if (wait || found)
                continue;
            if (__ballot(w[i] < CHAIN_SUM)) { // one is not published yet
                wait = true;
                continue;
            }
            const u64 pre = __ballot(w[i] >= CHAIN_PREFIX);
            const int stop = pre ? (int)__builtin_ctzll(pre) : 63; // nearest prefix
            sum += wave_sum(lane <= stop ? w[i] & CHAIN_VALUE : 0ull);
            found = pre != 0;
            used += 64;
        }
        before += sum;
        if (found)
            break;
        e -= used;
        if (wait && !used)
            __builtin_amdgcn_s_sleep(1);
    }
    if (lane == 0 && b)
        device_store(&words[b], CHAIN_PREFIX | (before + part));
    return before;
}

// ---- B -> tiles ------------------------------------------------------------------------
//
// One pass over B's entries (a row of any length costs the same per entry: R-MAT's hub rows
// made a row-per-group conversion wait on its longest row).  A block takes BT_N consecutive
// entries; it finds the rows that start among them by searching the row pointers, marks
// their first entries in LDS, flags tile heads (first entry of a row, or another tile than
// the left neighbour's), counts them with ballots, learns the tiles before it from the
// chained scan, and writes its tiles and its rows' tile pointers.  A tile's bits are OR-ed
// in LDS by the block that holds its head, which reads on past its end for them.  Every
// block also validates a share of the row pointers.
// What bounds it: HBM (4 bytes read per entry, 12 written per tile) and, for small B, the
// latency of the search and the chain.  It takes the place of nine kernels (row marks, head
// flags, a three-kernel scan, fill, carry, tile pointers and a clear), which read the
// entries and the flags several times over.
// Reference: compute_tile64_nums / compute_tile64_col / compute_tile64_mask_num,
// src/compressed/compressed_mask64.cuh:61-342.
constexpr int BT_BS = 256;
constexpr int BT_STEPS = 8;                      // entries per thread
constexpr int BT_N = BT_BS * BT_STEPS;           // entries per block
constexpr int BT_WAVE = BT_N / (BT_BS / 64);     // entries per wave, 64 per step
static_assert(BT_WAVE == 64 * BT_STEPS, "a wave's entries are its steps");

// The first r in [0, n) with rp[r] >= x (n if none), for nondecreasing rp, by one wave: each
// round cuts the range to a 65th.  (Any rp: the result is some r in [0, n].)
DEVI int first_row(const int *__restrict__ rp, long long n, long long x)
{
    const int lane = threadIdx.x & 63;
    long long lo = 0, hi = n; // the answer lies in [lo, hi]
    while (hi > lo) {
        const long long step = (hi - lo + 63) / 64;
        const long long q = lo + lane * step;
        const bool ge = q >= hi || (long long)rp[q] >= x;
        const u64 m = __ballot(ge); // lanes from the first set one on (sorted rp)
        const int f = m ? (int)__builtin_ctzll(m) : 64;
        if (f == 0) {
            hi = lo;
        } else {
            const long long l2 = lo + (f - 1) * step + 1, h2 = lo + f * step;
            hi = h2 < hi ? h2 : hi;
            lo = l2;
        }
    }
    return (int)uniform64(lo);
}

__global__ __launch_bounds__(BT_BS) void k_btiles(int64_t K, int64_t N, int64_t nnz, const int *__restrict__ rp,
                                                  const int *__restrict__ col, int *__restrict__ tptr,
                                                  int *__restrict__ tcol, u64 *__restrict__ tmask,
                                                  BRow *__restrict__ brow, u64 *words, unsigned *ticket, DevStats *st)
{
    __shared__ u64 s_mask[BT_N]; // bits of the block's tiles
    __shared__ u64 s_start[BT_N / 64];
    __shared__ u64 s_head[BT_N / 64];
    __shared__ int s_before[BT_N / 64]; // heads before each 64 entries, within the block
    __shared__ int s_b, s_r0, s_r1, s_prefix, s_tiles;
    const int t = threadIdx.x, lane = t & 63, w = uniform(t >> 6);
    if (t == 0) // (a lone block has no place to take)
        s_b = gridDim.x > 1 ? (int)atomicAdd(ticket, 1u) : 0;
    for (int q = t; q < BT_N; q += BT_BS)
        s_mask[q] = 0;
    if (t < BT_N / 64)
        s_start[t] = 0;
    __syncthreads();
    const int b = uniform(s_b);
    const int nb = (int)gridDim.x;
    const int64_t e0 = (int64_t)b * BT_N;
    const int64_t e1 = e0 + BT_N < nnz ? e0 + BT_N : nnz;
    int bad = 0;
    // this block's share of the row pointers: in range and nondecreasing
    {
        const int64_t v0 = K * b / nb, v1 = K * (b + 1) / nb;
        for (int64_t r = v0 + t; r < v1; r += BT_BS) {
            const int s = rp[r], e = rp[r + 1];
            if (s < 0 || e < s || (int64_t)e > nnz)
                bad |= ERR_ROWPTR;
        }
    }
    // rows whose first entry is in [e0, e1): [r0, r1); the last block takes the rest
    if (w == 0) {
        const int r = first_row(rp, K + 1, e0);
        if (lane == 0)
            s_r0 = b == 0 ? 0 : r;
    } else if (w == 1) {
        const int r = first_row(rp, K + 1, e1);
        if (lane == 0)
            s_r1 = b == nb - 1 ? (int)(K + 1) : r;
    }
    // the wave's columns, and each one's left neighbour through the lanes
    int c[BT_STEPS], pc[BT_STEPS];
    const int64_t k0 = e0 + (int64_t)w * BT_WAVE;
#pragma unroll
    for (int i = 0; i < BT_STEPS; ++i) {
        const int64_t k = k0 + 64 * i + lane;
        c[i] = k < e1 ? col[k] : 0;
    }
    int carry = k0 > 0 && k0 < e1 ? col[k0 - 1] : 0;
#pragma unroll
    for (int i = 0; i < BT_STEPS; ++i) {
        pc[i] = __builtin_amdgcn_update_dpp(carry, c[i], 0x138, 0xf, 0xf, false); // wave_shr:1
        carry = __builtin_amdgcn_readlane(c[i], 63);
    }
    __syncthreads();
    const int r0 = uniform(s_r0), r1 = uniform(s_r1);
    for (int64_t r = (int64_t)r0 + t; r < r1; r += BT_BS) {
        const int64_t p = rp[r];
        if (p >= e0 && p < e1)
            atomicOr(&s_start[(p - e0) >> 6], 1ull << ((p - e0) & 63));
    }
    __syncthreads();
    u64 H[BT_STEPS];
#pragma unroll
    for (int i = 0; i < BT_STEPS; ++i) {
        const int64_t k = k0 + 64 * i + lane;
        const bool in = k < e1;
        const bool start = __builtin_amdgcn_inverse_ballot_w64(uniform64(s_start[w * BT_STEPS + i])) || k == 0;
        if (in && (unsigned)c[i] >= (unsigned long long)N)
            bad |= ERR_BCOL;
        if (in && !start && pc[i] > c[i])
            bad |= ERR_UNSORTED;
        H[i] = __ballot(in && (start || (pc[i] >> 6) != (c[i] >> 6)));
        if (lane == 0)
            s_head[w * BT_STEPS + i] = H[i];
    }
    if (bad)
        atomicOr(&st->err, bad);
    __syncthreads();
    // heads before each 64 entries, the block's tiles and the tiles before it
    if (w == 0) {
        static_assert(BT_N / 64 <= 64, "one wave scans the block's heads");
        const int n = lane < BT_N / 64 ? __popcll(s_head[lane]) : 0;
        const int incl = wave_incl_scan(n);
        if (lane < BT_N / 64)
            s_before[lane] = incl - n;
        const int tiles = wave_last(incl);
        const u64 pre = chain_prefix(words, b, (u64)tiles);
        if (lane == 0) {
            s_tiles = tiles;
            s_prefix = (int)pre;
        }
    }
    __syncthreads();
    const int prefix = uniform(s_prefix), tiles = uniform(s_tiles);
#pragma unroll
    for (int i = 0; i < BT_STEPS; ++i) {
        const int64_t k = k0 + 64 * i + lane;
        const bool head = __builtin_amdgcn_inverse_ballot_w64(H[i]);
        const int at = s_before[w * BT_STEPS + i] + mbcnt(H[i]) + (head ? 1 : 0) - 1; // this entry's tile
        if (k < e1 && at >= 0) // (before the first head: another block's tile)
            atomicOr(&s_mask[at], 1ull << (c[i] & 63));
        if (head)
            tcol[prefix + at] = c[i] >> 6;
    }
    // entries past the block that belong to its last tile: the same row and tile
    if (w == 0 && tiles > 0 && e1 < nnz) {
        const int64_t row_end = r1 <= K ? (int64_t)rp[r1] : nnz; // of the row of entry e1 - 1
        const int64_t end = row_end < nnz ? row_end : nnz;
        const int last = col[e1 - 1] >> 6;
        for (int64_t k = e1 + lane;; k += 64) {
            const int cc = k < end ? col[k] : 0;
            const bool mine = k < end && (cc >> 6) == last;
            if (mine)
                atomicOr(&s_mask[tiles - 1], 1ull << (cc & 63));
            if (__ballot(mine) != ~0ull)
                break;
        }
    }
    // the block's rows: tiles before entry p of this block
    for (int64_t r = (int64_t)r0 + t; r < r1; r += BT_BS) {
        const int64_t p = rp[r];
        if (p < e0 || p > e1 || (p == e1 && e1 < nnz))
            continue; // (row pointers out of order: reported)
        int tp = tiles;
        if (p < e1) {
            const int q = (int)(p - e0);
            tp = s_before[q >> 6] + __popcll(s_head[q >> 6] & below(q & 63));
        }
        tp += prefix;
        tptr[r] = tp;
        if (r == K) {
            st->ntiles_b = tp;
        } else if (brow) {
            const int64_t e = rp[r + 1];
            BRow q = {0, 0, INT_MAX, -1};
            if (e > p && e <= nnz) { // rows are sorted: their first and last tiles
                q.len = (int)(e - p);
                q.ntiles = -1; // known if the row ends in this block
                if (e < e1) {
                    const int f = (int)(e - e0);
                    q.ntiles = prefix + s_before[f >> 6] + __popcll(s_head[f >> 6] & below(f & 63)) - tp;
                } else if (e == e1) {
                    q.ntiles = prefix + tiles - tp;
                }
                q.first = col[p] >> 6;
                q.last = col[e - 1] >> 6;
            }
            brow[r] = q;
        }
    }
    __syncthreads();
    for (int q = t; q < tiles; q += BT_BS)
        tmask[prefix + q] = s_mask[q];
}

int64_t btiles_blocks(int64_t nnz) { return nnz > 0 ? (nnz + BT_N - 1) / BT_N : 1; }

hipError_t launch_btiles(int64_t K, int64_t N, int64_t nnz, const int *rp, const int *col, int *tptr, int *tcol,
                         u64 *tmask, BRow *brow, u64 *words, unsigned *ticket, DevStats *st, hipStream_t s)
{
    hipLaunchKernelGGL(k_btiles, dim3((unsigned)btiles_blocks(nnz)), dim3(BT_BS), 0, s, K, N, nnz, rp, col, tptr, tcol,
                       tmask, brow, words, ticket, st);
    return hipGetLastError();
}

// ---- B's rows without their tiles -----------------------------------------------------------
//
// The records of B's rows (length, tiles, first and last tile) and the checks of k_btiles,
// for a B of short rows: rows of C that share a wave read B itself, so the tiles are made
// only once a row turns out to want them.  8 lanes per row, BR_U rows at a time; rows of
// more than BR_LONG entries a wave each, of more than BR_BLOCK the block.  Bound by the
// chain row pointer -> columns; 45 M entries in 7.5 M rows take 180 us, their tiles 477.
constexpr int BR_BS = 256;
constexpr int BR_G = 8;
constexpr int BR_U = 4;
constexpr int BR_ROWS = 256; // rows of a block at a time
constexpr int BR_LONG = 64;
constexpr int BR_BLOCK = 16384;

__global__ __launch_bounds__(BR_BS) void k_brows(int64_t K, int64_t N, int64_t nnz, const int *__restrict__ rp,
                                                 const int *__restrict__ col, BRow *__restrict__ brow, DevStats *st)
{
    __shared__ int s_long, s_tiles, s_part;
    __shared__ unsigned short s_list[BR_ROWS];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, g = t / BR_G, l = t & (BR_G - 1);
    int bad = 0, total = 0; // tiles counted by this thread
    // entry k of a row from s: is it its tile's first?
    auto head = [&](int64_t k, int64_t s, int c, int before) {
        if ((unsigned)c >= (unsigned long long)N)
            bad |= ERR_BCOL;
        if (k > s && before > c)
            bad |= ERR_UNSORTED;
        return k == s || (before >> 6) != (c >> 6) ? 1 : 0;
    };
    auto store = [&](int64_t r, int s, int e, int tiles, int c0, int c1) {
        brow[r] = e > s ? BRow{e - s, tiles, c0 >> 6, c1 >> 6} : BRow{0, 0, INT_MAX, -1};
    };
    if (blockIdx.x == 0) { // entries of no row (row pointers that do not start at 0 or end at nnz)
        const int64_t a = rp[0] < nnz ? rp[0] : nnz, b = rp[K] > 0 ? rp[K] : 0;
        for (int64_t k = t; k < a; k += BR_BS)
            (void)head(k, 0, col[k], k > 0 ? col[k - 1] : 0);
        for (int64_t k = b + t; k < nnz; k += BR_BS)
            (void)head(k, 0, col[k], k > 0 ? col[k - 1] : 0);
    }
    if (t == 0)
        s_tiles = 0;
    for (int64_t i0 = (int64_t)blockIdx.x * BR_ROWS; i0 < K; i0 += (int64_t)gridDim.x * BR_ROWS) {
        const int n = (int)(K - i0 < BR_ROWS ? K - i0 : BR_ROWS);
        if (t == 0)
            s_long = 0;
        __syncthreads();
        for (int q0 = g; q0 < n; q0 += BR_U * (BR_BS / BR_G)) {
            int s[BR_U], e[BR_U], c[BR_U];
#pragma unroll
            for (int u = 0; u < BR_U; ++u) {
                const int q = q0 + u * (BR_BS / BR_G);
                s[u] = e[u] = 0;
                if (q < n) {
                    s[u] = rp[i0 + q];
                    e[u] = rp[i0 + q + 1];
                }
            }
#pragma unroll
            for (int u = 0; u < BR_U; ++u) {
                if (s[u] < 0 || e[u] < s[u] || (int64_t)e[u] > nnz) {
                    bad |= ERR_ROWPTR;
                    e[u] = s[u] = 0;
                }
                c[u] = s[u] + l < e[u] && e[u] - s[u] <= BR_LONG ? col[s[u] + l] : 0;
            }
#pragma unroll
            for (int u = 0; u < BR_U; ++u) {
                const int q = q0 + u * (BR_BS / BR_G);
                const bool lng = e[u] - s[u] > BR_LONG;
                const int before = __builtin_amdgcn_update_dpp(0, c[u], 0x138, 0xf, 0xf, false); // wave_shr:1
                int sum = 0, last = c[u]; // (sorted: the largest)
                if (!lng) {
                    if (s[u] + l < e[u])
                        sum = head(s[u] + l, s[u], c[u], before);
                    for (int k = s[u] + l + BR_G; k < e[u]; k += BR_G) {
                        const int cc = col[k];
                        sum += head(k, s[u], cc, col[k - 1]);
                        last = cc;
                    }
                    total += sum;
                }
                sum = group_sum<BR_G>(sum);
                last = group_max<BR_G>(last);
                if (l == 0 && q < n) {
                    if (lng)
                        s_list[atomicAdd(&s_long, 1)] = (unsigned short)q;
                    else
                        store(i0 + q, s[u], e[u], sum, c[u], last);
                }
            }
        }
        __syncthreads();
        const int nlong = s_long;
        for (int i = 0; i < nlong; ++i) {
            const int q = s_list[i];
            const int s = rp[i0 + q], e = rp[i0 + q + 1];
            const bool block = e - s > BR_BLOCK; // (the same in every thread)
            if (!block && (i & (BR_BS / 64 - 1)) != w)
                continue;
            int sum = 0;
#pragma unroll 4
            for (int64_t k = (int64_t)s + (block ? t : lane); k < e; k += block ? BR_BS : 64)
                sum += head(k, s, col[k], k > s ? col[k - 1] : 0);
            total += sum;
            sum = wave_sum(sum);
            if (!block) {
                if (lane == 0)
                    store(i0 + q, s, e, sum, col[s], col[e - 1]);
                continue;
            }
            if (t == 0)
                s_part = 0;
            __syncthreads();
            if (lane == 0)
                atomicAdd(&s_part, sum);
            __syncthreads();
            if (t == 0)
                store(i0 + q, s, e, s_part, col[s], col[e - 1]);
            __syncthreads();
        }
        __syncthreads();
    }
    if (bad)
        atomicOr(&st->err, bad);
    total = wave_sum(total);
    __syncthreads();
    if (lane == 0)
        atomicAdd(&s_tiles, total);
    __syncthreads();
    if (t == 0 && s_tiles)
        atomicAdd(&st->ntiles_b, s_tiles);
}

hipError_t launch_brows(int64_t K, int64_t N, int64_t nnz, const int *rp, const int *col, BRow *brow, DevStats *st,
                        int num_cus, hipStream_t s)
{
    const int64_t chunks = (K + BR_ROWS - 1) / BR_ROWS, most = 32 * (int64_t)num_cus;
    hipLaunchKernelGGL(k_brows, dim3((unsigned)(chunks < 1 ? 1 : chunks < most ? chunks : most)), dim3(BR_BS), 0, s, K, N,
                       nnz, rp, col, brow, st);
    return hipGetLastError();
}

// ---- binning -----------------------------------------------------------------------------

// Bin of one row: lanes from work (per_lane items per lane, 8..1024 lanes), then fewer
// rows per workgroup until the workgroup's LDS fits the budget; rows whose own need
// exceeds row_max go to the global-memory bin.  need(b): the row's LDS in bin b.
// Reference ranges being replaced: src/bining.cuh:12 (symbolic), :121 (tile OR), :228
// (numeric).
// Lanes per row: the stream that rows with a workgroup of their own walk costs about the
// same per item at every width from 64 lanes, and a start and an end per row that narrow
// groups spread over more rows, so a lane gets 32 tiles or 48 products by default (symbolic
// stage at 4 / 16 / 32 tiles per lane: R-MAT squares of scale 16 746 / 476 / 439 us and of
// scale 18 6.67 / 4.28 / 3.52 ms, banded rows of 100 tiles 116 / 72 / 66 us; numeric bins at
// 32 / 48 / 64 / 96 products: banded rows of 4,096 products 553 / 483 / 484 us, R-MAT scale 15
// 681 / 658 / 662 / 690).  Rows whose
// elements fit the registers of 8, 16 or 32 lanes share a wave.  16 waves per CU, where LDS
// limits the workgroups, take 17.8 ms on the square of scale 18 against 19.2 ms with 8; 24
// slow a banded square by 4%.
// (nd: the row's need in the bin chosen)
template <typename Need>
DEVI int choose_bin(long long work, Need need, int row_max, const BinParams &bp, int &nd)
{
    int b = bp.force_global ? BIN_GLOBAL : 0;
    while (b < NLDS - 1 && (8LL << b) * bp.per_lane < work)
        ++b;
    nd = need(b);
    // the budget limits only workgroups that pack several rows: a one-row workgroup needs
    // the row's LDS whatever its width
    while (b < BIN_SHARED) {
        if (nd <= row_max && nd * (BLOCK >> (b + 3)) <= (b < BIN_SHARED - 1 ? bp.lds_block_budget : bp.lds_pair_budget))
            return b;
        nd = need(++b);
    }
    // a one-row workgroup's LDS decides how many fit a CU: widen the row's group until
    // those workgroups hold min_waves waves, to hide the latency of the gathers from B
    while (b < NLDS - 1) {
        const int waves = (8 << b) / 64, wgs = (bp.min_waves + waves - 1) / waves;
        if ((long long)nd * wgs <= bp.lds_cu)
            break;
        const int wider = need(b + 1);
        if (wider > row_max)
            break; // (the stream's tables grow a little with the width)
        nd = wider;
        ++b;
    }
    if (b < BIN_GLOBAL && nd > row_max) {
        b = BIN_GLOBAL;
        nd = need(b);
    }
    return b;
}

// One row as the binning sees it.
struct BinRow {
    long long prod;
    int S, nA, tp, nc; // tiles spanned, entries of A, tile-products, entries of C
};

// The blocks of one binning: their counts in LDS, then one global atomic per bin and block
// for the rows' places (atomics on one address retire one every few nanoseconds
// device-wide: with one more for each sum and maximum they were the binning's whole time).
// The sums and maxima go to one of BIN_PARTS parts, and the last block to finish adds those
// up and, given `host`, writes the totals there.  (With a part of its own for every block,
// that last addition kept a batch of 7.5 M rows waiting for 130 us, in each of the phases.)
struct BinBlock {
    int cnt[NBINS], need[NBINS], span[NBINS], base[NBINS], sparse[NBINS], na_max[NBINS];
    u64 work[NBINS], nc[NBINS], na[NBINS];
    u64 dir, dir_base;
    int last;
};

DEVI void bin_clear(BinBlock &B)
{
    const int t = threadIdx.x;
    if (t < NBINS) {
        B.cnt[t] = B.need[t] = B.span[t] = B.sparse[t] = B.na_max[t] = 0;
        B.work[t] = B.nc[t] = B.na[t] = 0;
    }
    if (t == 0)
        B.dir = 0;
}

// Where one of the block's rows goes.
struct BinPlace {
    int b = -1, pos = 0;
    long long dloc = -1;
};

// One row per lane of a wave (every lane of the wave calls it; r.prod == 0: no row).
DEVI BinPlace bin_row(BinBlock &B, int numeric, const BinRow &r, const BinParams &bp, DevStats *st)
{
    BinPlace at;
    int sp = 0;
    bool wide = false;
    long long work = 0;
    int need = 0, E = 0;
    if (r.prod > 0) {
        if (numeric) {
            work = r.prod;
            auto nd = [&](int bin) { return num_need(bin, r.S, r.nc, r.nA, r.tp, r.prod); };
            const bool giant = r.prod >= bp.giant_min && wide_hot(r.prod, r.nc, r.nA);
            at.b = choose_bin(work, nd, giant ? 0 : window_filled(r.nc, r.S) ? bp.lds_window_max : bp.lds_row_max, bp,
                              need);
        } else {
            work = r.tp;
            // the numeric need with nnz(C_i) <= min(products, 64 * span): a row that may be wide
            // there keeps a directory, which rows that share a wave do not make
            const long long nub = r.prod < 64LL * r.S ? r.prod : 64LL * r.S;
            const int most = bp.lds_row_max < WINDOW_ROW_MIN ? bp.lds_row_max : WINDOW_ROW_MIN;
            wide = num_need(NLDS - 1, r.S, (int)(nub < INT_MAX ? nub : INT_MAX), r.nA, r.tp, r.prod) > most;
            auto nd = [&](int bin) {
                return wide && bin < BIN_SHARED ? LAYOUT_NONE : sym_need(bin, r.S, r.nA, r.tp, r.prod);
            };
            at.b = choose_bin(work, nd, bp.lds_row_max, bp, need);
            // directory entries kept for the numeric phase: the row's form in an LDS bin, the
            // flat span for rows the symbolic phase handles in global memory
            E = at.b < BIN_SHARED ? 0 : at.b < BIN_GLOBAL ? dir_entries(r.S, r.tp) : r.S;
        }
        sp = use_sparse(r.S, r.tp) ? 1 : 0;
    }
    const int lane = threadIdx.x & 63;
    if (__ballot(wide)) {
        const u64 products = wave_sum(wide ? (u64)r.prod : 0ull);
        if (lane == 0)
            atomicAdd(&st->num_wide_work, products);
    }
    if (!numeric && __ballot(r.prod > (long long)WIDE_GIANT)) {
        const u64 most = wave_most((u64)r.prod);
        if (lane == 0)
            atomicMax(&st->prod_most, most);
    }
    if (numeric && __ballot(at.b == BIN_GLOBAL)) { // room for the wide rows' windows
        const u64 mine = at.b == BIN_GLOBAL ? (u64)wide_row_items(r.nc, r.S) : 0ull;
        const u64 items = wave_sum(mine);
        if (lane == 0)
            atomicAdd(&st->wide_items, items);
        const bool hot = at.b == BIN_GLOBAL && wide_hot(r.prod, r.nc, r.nA);
        if (__ballot(hot)) {
            const u64 hots = wave_sum(hot ? mine : 0ull);
            const u64 most = wave_most(hot ? (u64)(r.prod - r.nc) : 0ull);
            if (lane == 0) {
                atomicAdd(&st->hot_items, hots);
                atomicMax(&st->hot_most, most);
            }
        }
    }
    // the lanes that chose one bin (neighbouring rows usually share it) add up first
    u64 pending = __ballot(at.b >= 0);
    while (pending) {
        const int leader = (int)__builtin_ctzll(pending);
        const int bb = __builtin_amdgcn_readlane(at.b, leader);
        const bool mine = at.b == bb;
        const u64 same = __ballot(mine);
        pending &= ~same;
        const u64 wsum = wave_sum(mine ? (u64)work : 0ull);
        const u64 nas = wave_sum(mine ? (u64)r.nA : 0ull);
        const u64 ncs = wave_sum(mine ? (numeric ? (u64)r.nc : (u64)r.prod) : 0ull);
        const int needm = wave_max(mine ? need : 0);
        const int spanm = wave_max(mine ? r.S : 0);
        const int nam = wave_max(mine ? r.nA : 0);
        const int sps = (int)__popcll(__ballot(mine && sp));
        const u64 dincl = numeric ? 0ull : wave_incl_scan(mine ? (u64)E : 0ull);
        const u64 dtot = numeric ? 0ull : wave_last(dincl);
        int base = 0;
        u64 dbase = 0;
        if (lane == leader) {
            base = atomicAdd(&B.cnt[bb], (int)__popcll(same));
            atomicMax(&B.need[bb], needm);
            atomicMax(&B.span[bb], spanm);
            atomicMax(&B.na_max[bb], nam);
            atomicAdd(&B.work[bb], wsum);
            atomicAdd(&B.na[bb], nas);
            atomicAdd(&B.nc[bb], ncs);
            if (sps)
                atomicAdd(&B.sparse[bb], sps);
            if (dtot)
                dbase = atomicAdd(&B.dir, dtot);
        }
        base = __builtin_amdgcn_readlane(base, leader);
        dbase = readlane_u64(dbase, leader);
        if (mine) {
            at.pos = base + mbcnt(same);
            if (E > 0)
                at.dloc = ((long long)(dbase + dincl) - E) | (sp && bb < BIN_GLOBAL ? RDIR_TWO : 0);
        }
    }
    return at;
}

// Reserve the places of the block's rows (every thread of the block; after a barrier).
DEVI void bin_reserve(BinBlock &B, int numeric, DevStats *st, BinSum *sums)
{
    const int t = threadIdx.x;
    BinStats *bs = numeric ? &st->num : &st->sym;
    if (t < NBINS) {
        const int c = B.cnt[t];
        B.base[t] = c ? atomicAdd(&bs->count[t], c) : 0;
        if (c && gridDim.x > 1) {
            BinSum *s = sums + (blockIdx.x % BIN_PARTS) * NBINS + t;
            atomicAdd(&s->work, B.work[t]);
            atomicAdd(&s->nnz_a, B.na[t]);
            atomicAdd(&s->nnz_c, B.nc[t]);
            atomicMax(&s->need, (unsigned)B.need[t]);
            atomicMax(&s->span, (unsigned)B.span[t]);
            atomicMax(&s->na_max, (unsigned)B.na_max[t]);
            if (B.sparse[t])
                atomicAdd(&s->nsparse, (unsigned)B.sparse[t]);
        }
    }
    if (!numeric && t == NBINS)
        B.dir_base = B.dir ? atomicAdd(&st->dir_total, B.dir) : 0;
    __syncthreads();
}

// The end of a binning: the last block adds the blocks' sums up and hands the counters to
// the host.  Every thread of the block (of blockDim.x >= NBINS).
DEVI void bin_finish(BinBlock &B, int numeric, DevStats *st, const BinSum *sums, unsigned *done, HostStats *host,
                     unsigned seq)
{
    const int t = threadIdx.x;
    const int nblk = (int)gridDim.x;
    if (nblk > 1) {
        // each thread's own updates are done (at the device's point of coherence: no cache
        // has to be written back)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (t == 0)
            B.last = atomicAdd(done, 1u) == (unsigned)nblk - 1;
        __syncthreads();
        if (!B.last)
            return;
        bin_clear(B);
        __syncthreads();
        static_assert(BIN_PARTS * NBINS <= 256, "a thread per part and bin");
        if (t < BIN_PARTS * NBINS) {
            const int bin = t % NBINS;
            const BinSum *s = sums + t;
            atomicAdd(&B.work[bin], device_load(&s->work));
            atomicAdd(&B.nc[bin], device_load(&s->nnz_c));
            atomicAdd(&B.na[bin], device_load(&s->nnz_a));
            atomicMax(&B.need[bin], (int)device_load(&s->need));
            atomicMax(&B.span[bin], (int)device_load(&s->span));
            atomicMax(&B.na_max[bin], (int)device_load(&s->na_max));
            atomicAdd(&B.sparse[bin], (int)device_load(&s->nsparse));
        }
        __syncthreads();
    }
    BinStats *bs = numeric ? &st->num : &st->sym;
    if (t < NBINS) {
        device_store(&bs->work[t], B.work[t]);
        device_store(&bs->nnz_c[t], B.nc[t]);
        device_store(&bs->nnz_a[t], B.na[t]);
        device_store(&bs->max_need[t], B.need[t]);
        device_store(&bs->max_span[t], B.span[t]);
        device_store(&bs->max_na[t], B.na_max[t]);
        device_store(&bs->nsparse[t], B.sparse[t]);
    }
    if (!host)
        return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // the counters arrive before the number that follows them: the host, which waits for it,
    // goes on without the end of the kernel
    const unsigned *from = (const unsigned *)st;
    unsigned *to = (unsigned *)&host->st;
    for (unsigned q = t; q < sizeof(DevStats) / sizeof(unsigned); q += blockDim.x)
        __hip_atomic_store(&to[q], device_load(&from[q]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t == 0)
        __hip_atomic_store(&host->seq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---- row analysis of A ---------------------------------------------------------------

// Per row i of A: products sum_j nnz(B_j), tile-products sum_j tiles(B_j), and the span
// [rmin, rmax] of tile columns of row i of C (rows of B are sorted, so each B row's first
// and last tile bound it); then the symbolic binning of the block's rows.  Reference:
// k_compute_flop, src/small/mask.cuh:14-51.
// A group of G lanes per row; a block takes `rows` rows, a lane group each at a time, and bins them
// together, so that the binning's atomics are few and hide behind other blocks' gathers.
// Rows of more than LONG_A entries per lane are listed and left to whole waves, those of
// more than LONG_WAVE entries to the whole block (at 2,048 entries for every group width,
// a hub row's 16 lanes kept an R-MAT graph's analysis waiting).
constexpr int LONG_A = 16;
constexpr int LONG_WAVE = 4096;
// Short rows (G = 8) take blocks of 512 lanes, of which twice as many overlap on a CU, and at
// least 128 rows each, as more blocks queue at the bins' counters: 7.5 M rows of 6 entries
// take 464 us with 1,024 lanes and 330 with 512, 16,384 rows 10.8 and, with 64 rows per
// block, 11.6.  Longer rows gather more per row: an R-MAT graph of scale 18 takes 383 us with
// 1,024 lanes and 595 with 512.
constexpr int ri_lanes(int G) { return G == 8 ? 512 : 1024; }
constexpr int ri_rows_max(int G) { return 2 * ri_lanes(G); } // rows of a block

template <int G>
__global__ __launch_bounds__(ri_lanes(G)) void k_row_info(int64_t M, int64_t K, int64_t nnzA, int rows,
                                                  const int *__restrict__ Arp, const int *__restrict__ Acol,
                                                  const BRow *__restrict__ brow, const int *__restrict__ tptr,
                                                  long long *__restrict__ rprod, int *__restrict__ rtp, int *__restrict__ rmin,
                                                  int *__restrict__ rmax, int *__restrict__ rnnz, BinParams bp,
                                                  int *__restrict__ binrows, long long *__restrict__ rdir,
                                                  DevStats *st, BinSum *sums, unsigned *done, HostStats *host, unsigned seq)
{
    constexpr int RI_BS = ri_lanes(G), ROWS_MAX = ri_rows_max(G), RPB = RI_BS / G, NW = RI_BS / 64;
    __shared__ long long s_prod[ROWS_MAX];
    __shared__ int s_tp[ROWS_MAX], s_mn[ROWS_MAX], s_mx[ROWS_MAX];
    __shared__ BinBlock B;
    __shared__ long long s_p[NW];
    __shared__ int s_t[NW], s_n[NW], s_x[NW];
    __shared__ int s_long;
    __shared__ unsigned short s_list[ROWS_MAX];
    const int t = threadIdx.x, g = t / G, l = t & (G - 1);
    const int64_t i0 = (int64_t)blockIdx.x * rows;
    const int n = (int)(M - i0 < rows ? M - i0 : rows);
    int bad = 0;
    bin_clear(B);
    if (t == 0)
        s_long = 0;
    __syncthreads();
    auto entry = [&](int j, long long &p, int &tp, int &mn, int &mx) {
        if ((unsigned)j >= (unsigned long long)K) {
            bad |= ERR_ACOL;
            return;
        }
        const BRow q = brow[j];
        p += q.len;
        tp += q.ntiles >= 0 ? q.ntiles : tptr[j + 1] - tptr[j];
        mn = q.first < mn ? q.first : mn;
        mx = q.last > mx ? q.last : mx;
    };
    // RU rows per group at a time: their dependent loads (row extent, column, record of B's
    // row) are issued together
    constexpr int RU = 4;
    for (int q0 = g; q0 < n; q0 += RU * RPB) {
        int s[RU], e[RU], tp[RU], mn[RU], mx[RU];
        long long p[RU];
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const int q = q0 + u * RPB;
            s[u] = e[u] = 0;
            if (q < n) {
                s[u] = Arp[i0 + q];
                e[u] = Arp[i0 + q + 1];
            }
        }
        int j[RU];
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            p[u] = 0;
            tp[u] = 0;
            mn[u] = INT_MAX;
            mx[u] = -1;
            if (s[u] < 0 || e[u] < s[u] || (int64_t)e[u] > nnzA) {
                bad |= ERR_ROWPTR;
                e[u] = s[u] = 0;
            } else if (e[u] - s[u] > LONG_A * G) {
                if (l == 0)
                    s_list[atomicAdd(&s_long, 1)] = (unsigned short)(q0 + u * RPB);
                e[u] = s[u];
            }
            j[u] = s[u] + l < e[u] ? Acol[s[u] + l] : -1;
        }
#pragma unroll
        for (int u = 0; u < RU; ++u)
            if (s[u] + l < e[u])
                entry(j[u], p[u], tp[u], mn[u], mx[u]);
#pragma unroll
        for (int u = 0; u < RU; ++u)
            for (int k = s[u] + l + G; k < e[u]; k += G)
                entry(Acol[k], p[u], tp[u], mn[u], mx[u]);
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const int q = q0 + u * RPB;
            const long long ps = group_sum<G>(p[u]);
            const int ts = group_sum<G>(tp[u]), ms = group_min<G>(mn[u]), xs = group_max<G>(mx[u]);
            if (q < n && l == 0) {
                s_prod[q] = ps;
                s_tp[q] = ts;
                s_mn[q] = ms;
                s_mx[q] = xs;
            }
        }
    }
    __syncthreads();
    const int nlong = s_long;
    for (int i = t >> 6; i < nlong; i += NW) { // listed rows: a wave each
        const int q = s_list[i], lane = t & 63;
        const int s = Arp[i0 + q], e = Arp[i0 + q + 1];
        if (e - s > LONG_WAVE)
            continue;
        long long p = 0;
        int tp = 0, mn = INT_MAX, mx = -1;
#pragma unroll 4
        for (int k = s + lane; k < e; k += 64)
            entry(Acol[k], p, tp, mn, mx);
        p = wave_sum(p);
        tp = wave_sum(tp);
        mn = group_min<64>(mn);
        mx = group_max<64>(mx);
        if (lane == 0) {
            s_prod[q] = p;
            s_tp[q] = tp;
            s_mn[q] = mn;
            s_mx[q] = mx;
        }
    }
    for (int i = 0; i < nlong; ++i) { // the longest: the block each
        const int q = s_list[i];
        const int s = Arp[i0 + q], e = Arp[i0 + q + 1];
        if (e - s <= LONG_WAVE)
            continue;
        long long p = 0;
        int tp = 0, mn = INT_MAX, mx = -1;
#pragma unroll 4
        for (int k = s + t; k < e; k += RI_BS)
            entry(Acol[k], p, tp, mn, mx);
        p = wave_sum(p);
        tp = wave_sum(tp);
        mn = group_min<64>(mn);
        mx = group_max<64>(mx);
        if ((t & 63) == 0) {
            s_p[t >> 6] = p;
            s_t[t >> 6] = tp;
            s_n[t >> 6] = mn;
            s_x[t >> 6] = mx;
        }
        __syncthreads();
        if (t == 0) {
            for (int w = 1; w < NW; ++w) {
                p += s_p[w];
                tp += s_t[w];
                mn = s_n[w] < mn ? s_n[w] : mn;
                mx = s_x[w] > mx ? s_x[w] : mx;
            }
            s_prod[q] = p;
            s_tp[q] = tp;
            s_mn[q] = mn;
            s_mx[q] = mx;
        }
        __syncthreads();
    }
    __syncthreads();
    if (bad)
        atomicOr(&st->err, bad);
    // the rows' values, and their bins
    BinPlace at[ROWS_MAX / RI_BS];
#pragma unroll
    for (int u = 0; u < ROWS_MAX / RI_BS; ++u) {
        if (u * RI_BS >= n) // uniform
            break;
        const int q = u * RI_BS + t;
        BinRow r = {0, 0, 0, 0, 0};
        if (q < n) {
            const int64_t i = i0 + q;
            const int mn = s_mn[q], mx = s_mx[q];
            r.prod = s_prod[q];
            r.S = mx - mn + 1;
            r.tp = s_tp[q];
            r.nA = Arp[i + 1] - Arp[i];
            rprod[i] = r.prod;
            rtp[i] = r.tp;
            rmin[i] = mn;
            rmax[i] = mx;
            if (r.prod == 0)
                rnnz[i] = 0;
        }
        at[u] = bin_row(B, 0, r, bp, st);
    }
    __syncthreads();
    bin_reserve(B, 0, st, sums);
#pragma unroll
    for (int u = 0; u < ROWS_MAX / RI_BS; ++u) {
        const int q = u * RI_BS + t;
        if (q >= n)
            break;
        if (at[u].b >= 0)
            binrows[(int64_t)at[u].b * M + B.base[at[u].b] + at[u].pos] = (int)(i0 + q);
        rdir[i0 + q] = at[u].dloc >= 0 ? (long long)B.dir_base + at[u].dloc : -1;
    }
    bin_finish(B, 0, st, sums, done, host, seq);
}

static int row_info_lanes(int64_t M, int64_t nnzA)
{
    const int64_t avg = nnzA / (M > 0 ? M : 1);
    return avg <= 12 ? 8 : (avg <= 24 ? 16 : (avg <= 48 ? 32 : 64));
}

// Rows per block: two blocks per CU hold all its waves; beyond that, as many rows as the
// block's LDS holds, for fewer atomics per row.
static int row_info_rows(int64_t M, int64_t nnzA, int num_cus)
{
    const int G = row_info_lanes(M, nnzA), rpb = ri_lanes(G) / G;
    const int64_t full = (int64_t)rpb * 2 * num_cus;
    const int64_t least = G == 8 ? 2 : 1, most = ri_rows_max(G) / rpb;
    const int64_t passes = (M + full - 1) / full;
    return (int)(passes < least ? least : passes > most ? most : passes) * rpb;
}

static int64_t row_info_blocks(int64_t M, int64_t nnzA, int num_cus)
{
    const int rows = row_info_rows(M, nnzA, num_cus);
    return (M + rows - 1) / rows;
}

hipError_t launch_row_info(int64_t M, int64_t K, int64_t nnzA, const int *Arp, const int *Acol, const BRow *brow,
                           const int *tptr, long long *rprod, int *rtp, int *rmin, int *rmax, int *rnnz, BinParams bp,
                           int *binrows, long long *rdir, DevStats *st, BinSum *sums, unsigned *done, HostStats *host,
                           unsigned seq,
                           int num_cus, hipStream_t s)
{
    const int rows = row_info_rows(M, nnzA, num_cus);
    const unsigned blocks = (unsigned)row_info_blocks(M, nnzA, num_cus);
#define ROW_INFO(G)                                                                                                    \
    case G:                                                                                                            \
        hipLaunchKernelGGL((k_row_info<G>), dim3(blocks), dim3(ri_lanes(G)), 0, s, M, K, nnzA, rows, Arp, Acol, brow, tptr,  \
                           rprod, rtp, rmin, rmax, rnnz, bp, binrows, rdir, st, sums, done, host, seq);                     \
        break;
    switch (row_info_lanes(M, nnzA)) {
        ROW_INFO(8) ROW_INFO(16) ROW_INFO(32) ROW_INFO(64)
    }
#undef ROW_INFO
    return hipGetLastError();
}

// C's row pointers from nnz(C_i) (chained scan) and the numeric binning, T rows per lane.
// out32 (may be null): the row pointers as int32 too, for the caller.  Each block takes a
// place, then places in the bins, and waits for the blocks before it, so many rows go two to
// a lane (7.5 M rows: 196 us with one, 172 with two); up to RP_FEW go one to a lane, on
// more CUs.
constexpr int RP_BS = 1024;
constexpr int RP_FEW = 1 << 19;

template <int T>
__global__ __launch_bounds__(RP_BS) void k_rowptr_bin(int64_t M, const int *__restrict__ Arp,
                                                    const long long *__restrict__ rprod, const int *__restrict__ rtp,
                                                    const int *__restrict__ rmin, const int *__restrict__ rmax,
                                                    const int *__restrict__ rnnz, long long *__restrict__ crp,
                                                    int *__restrict__ out32, BinParams bp, int *__restrict__ binrows,
                                                    u64 *words, unsigned *ticket, DevStats *st, BinSum *sums,
                                                    unsigned *done, HostStats *host, unsigned seq)
{
    __shared__ BinBlock B;
    __shared__ u64 red[RP_BS / 64];
    __shared__ u64 s_pre;
    __shared__ int s_b;
    const int t = threadIdx.x;
    bin_clear(B);
    if (t == 0)
        s_b = gridDim.x > 1 ? (int)atomicAdd(ticket, 1u) : 0;
    __syncthreads();
    const int b = uniform(s_b);
    const int64_t i0 = (int64_t)b * (T * RP_BS) + t;
    int nc[T];
    u64 pre[T], total = 0; // entries of the block's rows before this one's
#pragma unroll
    for (int u = 0; u < T; ++u)
        nc[u] = i0 + u * RP_BS < M ? rnnz[i0 + u * RP_BS] : 0;
#pragma unroll
    for (int u = 0; u < T; ++u) {
        u64 tot;
        pre[u] = total + group_excl_scan<RP_BS, u64>((u64)(unsigned)nc[u], red, tot);
        total += tot;
    }
    if (t < 64) {
        const u64 before = chain_prefix(words, b, total);
        if (t == 0)
            s_pre = before;
    }
    BinPlace at[T];
#pragma unroll
    for (int u = 0; u < T; ++u) {
        const int64_t i = i0 + u * RP_BS;
        BinRow r = {0, 0, 0, 0, 0};
        if (i < M) {
            r.prod = rprod[i];
            r.nc = nc[u];
            r.S = rmax[i] - rmin[i] + 1;
            r.nA = Arp[i + 1] - Arp[i];
            r.tp = rtp[i];
        }
        at[u] = bin_row(B, 1, r, bp, st);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < T; ++u) {
        const int64_t i = i0 + u * RP_BS;
        if (i < M) {
            const u64 at0 = s_pre + pre[u], end = at0 + (u64)(unsigned)nc[u];
            crp[i] = (long long)at0;
            if (out32)
                out32[i] = (int)at0;
            if (i == M - 1) {
                crp[M] = (long long)end;
                if (out32)
                    out32[M] = (int)end;
                device_store(&st->nnz_c, (long long)end);
            }
        }
    }
    bin_reserve(B, 1, st, sums);
#pragma unroll
    for (int u = 0; u < T; ++u)
        if (at[u].b >= 0)
            binrows[(int64_t)at[u].b * M + B.base[at[u].b] + at[u].pos] = (int)(i0 + u * RP_BS);
    bin_finish(B, 1, st, sums, done, host, seq);
}

int64_t rowptr_blocks(int64_t M)
{
    const int64_t rows = M > RP_FEW ? 2 * RP_BS : RP_BS;
    return (M + rows - 1) / rows;
}

hipError_t launch_rowptr_bin(int64_t M, const int *Arp, const long long *rprod, const int *rtp, const int *rmin,
                             const int *rmax, const int *rnnz, long long *crp, int *out32, BinParams bp, int *binrows,
                             u64 *words, unsigned *ticket, DevStats *st, BinSum *sums, unsigned *done, HostStats *host,
                             unsigned seq,
                             hipStream_t s)
{
    if (M <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(M > RP_FEW ? k_rowptr_bin<2> : k_rowptr_bin<1>, dim3((unsigned)rowptr_blocks(M)), dim3(RP_BS), 0,
                       s, M, Arp, rprod, rtp, rmin, rmax, rnnz, crp, out32, bp, binrows, words, ticket, st, sums, done,
                       host, seq);
    return hipGetLastError();
}

// ---- misc ------------------------------------------------------------------------------------

__global__ void k_pad_b(const int *col, const void *val, int val32, int n, int *pcol, void *pval)
{
    const int t = threadIdx.x;
    if (t >= STREAM_V)
        return;
    const int q = t < n ? t : n - 1;
    pcol[t] = col[q];
    if (val32)
        ((float *)pval)[t] = ((const float *)val)[q];
    else
        ((double *)pval)[t] = ((const double *)val)[q];
}

hipError_t launch_pad_b(const int *col, const void *val, int val32, int n, int *pcol, void *pval, hipStream_t s)
{
    hipLaunchKernelGGL(k_pad_b, dim3(1), dim3(64), 0, s, col, val, val32, n, pcol, pval);
    return hipGetLastError();
}

// ---- row pointers, row panels and row sums -------------------------------------------------

__global__ __launch_bounds__(256) void k_rowptr_narrow(const long long *__restrict__ in, int64_t n, int *__restrict__ out)
{
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        out[i] = (int)in[i];
}

hipError_t launch_rowptr_narrow(const long long *in, int64_t n, int *out, hipStream_t s)
{
    const int64_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(k_rowptr_narrow, dim3((unsigned)(blocks < 1 ? 1 : blocks < 8192 ? blocks : 8192)), dim3(256), 0, s,
                       in, n, out);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_rowptr_rebase(const int *__restrict__ in, int64_t n, int *__restrict__ out)
{
    const int base = in[0];
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        out[i] = in[i] - base;
}

hipError_t launch_rowptr_rebase(const int *in, int64_t n, int *out, hipStream_t s)
{
    int64_t blocks = (n + 255) / 256;
    blocks = blocks > 8192 ? 8192 : (blocks < 1 ? 1 : blocks);
    hipLaunchKernelGGL(k_rowptr_rebase, dim3((unsigned)blocks), dim3(256), 0, s, in, n, out);
    return hipGetLastError();
}

// One wave per row: sum and sum of magnitudes of the row's values.
template <typename RP, typename V>
__global__ __launch_bounds__(256) void k_row_sums(int64_t M, const RP *__restrict__ rp, const V *__restrict__ val,
                                                  double *__restrict__ sum, double *__restrict__ asum)
{
    const int lane = threadIdx.x & 63;
    const int64_t stride = (int64_t)gridDim.x * 4;
    for (int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); i < M; i += stride) {
        double s = 0.0, a = 0.0;
        for (long long k = (long long)rp[i] + lane; k < (long long)rp[i + 1]; k += 64) {
            const double v = (double)val[k];
            s += v;
            a += v < 0 ? -v : v;
        }
        s = wave_sum(s);
        a = wave_sum(a);
        if (lane == 0) {
            sum[i] = s;
            asum[i] = a;
        }
    }
}

hipError_t launch_row_sums(int64_t M, const void *rp, int rp64, const void *val, int val32, double *sum, double *asum,
                           hipStream_t s)
{
    int64_t blocks = (M + 3) / 4;
    blocks = blocks > 16384 ? 16384 : (blocks < 1 ? 1 : blocks);
    const dim3 g((unsigned)blocks), b(256);
    if (rp64 && val32)
        hipLaunchKernelGGL((k_row_sums<long long, float>), g, b, 0, s, M, (const long long *)rp, (const float *)val, sum, asum);
    else if (rp64)
        hipLaunchKernelGGL((k_row_sums<long long, double>), g, b, 0, s, M, (const long long *)rp, (const double *)val, sum,
                           asum);
    else if (val32)
        hipLaunchKernelGGL((k_row_sums<int, float>), g, b, 0, s, M, (const int *)rp, (const float *)val, sum, asum);
    else
        hipLaunchKernelGGL((k_row_sums<int, double>), g, b, 0, s, M, (const int *)rp, (const double *)val, sum, asum);
    return hipGetLastError();
}

// ---- batched form: stacking the instances and splitting C ----------------------------------

// Largest i in [0, count) with off[i] + i * step <= x (off nondecreasing, off[0] = 0 <= x):
// the instance whose range holds x, empty instances skipped.
DEVI int find_instance(const long long *__restrict__ off, int count, long long x, int step)
{
    int lo = 0, hi = count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] + (long long)mid * step <= x)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// The stacking kernels take chunks of STACK_CHUNK places per workgroup.  A chunk of few
// instances goes one instance after the other: the search for the first and the instance's
// fields are scalar, and a lane's loads need no lookup.  (A lookup per entry, stepping through
// the offsets in memory, kept 512 Laplacians' 45 M entries at 684 us for A and B, and a binary
// search per row their pointers at 75 us; now 252, one pass for both, and 20.)  In a chunk of
// more than STACK_FEW instances, where that is a chain of short waits, every lane finds its
// places' instances in a copy of the offsets in LDS: calls of 100,000 instances of 1 row 7.0 ms
// one after the other and 1.3 so, 20,000 of 9 rows 0.88 and 0.5, 4,000 of 64 rows 345 and 330 us,
// with 4, 16 or 64 as the limit.
// each(i, q, hi): this lane's places of instance i are q, q + 256, ... below hi.
constexpr int STACK_CHUNK = 4096;
constexpr int STACK_FEW = 16;
constexpr int STACK_U = 4; // loads in flight per lane
template <typename Each>
DEVI void stack_chunks(const long long *__restrict__ off, int step, int count, int64_t n, Each each)
{
    __shared__ unsigned short first[STACK_CHUNK]; // of the instances in the chunk, in it
    const int t = threadIdx.x;
    for (int64_t base = (int64_t)blockIdx.x * STACK_CHUNK; base < n; base += (int64_t)gridDim.x * STACK_CHUNK) {
        const int64_t end = base + STACK_CHUNK < n ? base + STACK_CHUNK : n;
        const int a = find_instance(off, count, base, step), more = a + STACK_FEW;
        if (more >= count || off[more] + (int64_t)more * step >= end) {
            for (int i = a; i < count; ++i) {
                const int64_t i0 = off[i] + (int64_t)i * step, i1 = off[i + 1] + (int64_t)(i + 1) * step;
                if (i0 >= end)
                    break;
                each(i, (i0 > base ? i0 : base) + t, i1 < end ? i1 : end);
            }
            continue;
        }
        const int b = find_instance(off, count, end - 1, step);
        const bool fit = b - a < STACK_CHUNK; // (more only with empty instances among them)
        if (fit) {
            __syncthreads();
            for (int i = t; i <= b - a; i += 256) // (the first starts at the chunk's start or before)
                first[i] = (unsigned short)(i ? off[a + i] + (int64_t)(a + i) * step - base : 0);
            __syncthreads();
        }
        for (int64_t q = base + t; q < end; q += 256) {
            int i = a;
            if (fit) {
                int lo = 0, hi = b - a; // the last instance that starts at q or before
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (first[mid] <= (unsigned)(q - base))
                        lo = mid;
                    else
                        hi = mid - 1;
                }
                i += lo;
            } else {
                i = find_instance(off, count, q, step);
            }
            each(i, q, q + 1);
        }
    }
}

__global__ __launch_bounds__(256) void k_batch_rowptr(int which, int count, const BatchInst *__restrict__ inst,
                                                      const long long *__restrict__ roff,
                                                      const long long *__restrict__ eoff, int64_t nrows, int64_t nnz,
                                                      int *__restrict__ out, DevStats *st)
{
    stack_chunks(roff, 0, count, nrows, [&](int i, int64_t q, int64_t hi) {
        const BatchInst &I = inst[i];
        const int64_t r0 = roff[i];
        const int *__restrict__ rp = (which ? I.Brp : I.Arp) - r0;
        const int e0 = (int)eoff[i];
        for (int64_t g = q; g < hi; g += 256)
            out[g] = e0 + rp[g];
        if (q == r0 && q < hi && // the instance's first row
            (rp[r0] != 0 || (long long)rp[r0 + (which ? I.K : I.M)] != eoff[i + 1] - eoff[i]))
            atomicOr(&st->err, ERR_ROWPTR);
    });
    if (blockIdx.x == 0 && threadIdx.x == 0)
        out[nrows] = (int)nnz;
}

template <typename T>
DEVI void copy_entries(const T *__restrict__ src, T *__restrict__ dst, int64_t q, int64_t hi)
{
    for (int64_t e = q; e < hi; e += STACK_U * 256) {
        T v[STACK_U];
#pragma unroll
        for (int u = 0; u < STACK_U; ++u)
            if (e + u * 256 < hi)
                v[u] = src[e + u * 256];
#pragma unroll
        for (int u = 0; u < STACK_U; ++u)
            if (e + u * 256 < hi)
                dst[e + u * 256] = v[u];
    }
}

__global__ __launch_bounds__(256) void k_batch_entries(int which, int count, const BatchInst *__restrict__ inst,
                                                       const long long *__restrict__ eoff,
                                                       const long long *__restrict__ koff, int64_t nnz, int val32,
                                                       int *__restrict__ Acol, int *__restrict__ Bcol,
                                                       void *__restrict__ val, DevStats *st)
{
    int bad = 0;
    stack_chunks(eoff, 0, count, nnz, [&](int i, int64_t q, int64_t hi) {
        const BatchInst &I = inst[i];
        const int64_t e0 = eoff[i];
        const int *__restrict__ src = (which ? I.Bcol : I.Acol) - e0;
        const int K = I.K, N = I.N, k0 = (int)koff[i];
        for (int64_t e = q; e < hi; e += STACK_U * 256) {
            int c[STACK_U];
#pragma unroll
            for (int u = 0; u < STACK_U; ++u)
                c[u] = e + u * 256 < hi ? src[e + u * 256] : 0;
#pragma unroll
            for (int u = 0; u < STACK_U; ++u) {
                if (e + u * 256 >= hi)
                    continue;
                if (Bcol) {
                    const bool in = (unsigned)c[u] < (unsigned)N;
                    bad |= in ? 0 : ERR_BCOL;
                    Bcol[e + u * 256] = in ? c[u] : 0;
                }
                if (Acol) {
                    const bool in = (unsigned)c[u] < (unsigned)K;
                    bad |= in ? 0 : ERR_ACOL;
                    Acol[e + u * 256] = (in ? c[u] : 0) + k0;
                }
            }
        }
        const void *from = which ? I.Bval : I.Aval;
        if (val32)
            copy_entries((const float *)from - e0, (float *)val, q, hi);
        else
            copy_entries((const double *)from - e0, (double *)val, q, hi);
    });
    if (bad)
        atomicOr(&st->err, bad);
}

__global__ __launch_bounds__(256) void k_batch_split(int count, const long long *__restrict__ mo,
                                                     const long long *__restrict__ crp, void *__restrict__ out,
                                                     int rp64, long long *__restrict__ bases)
{
    // C_i's M_i + 1 pointers lie from mo[i] + i
    stack_chunks(mo, 1, count, mo[count] + count, [&](int i, int64_t first, int64_t hi) {
        const long long *__restrict__ rp = crp - i;
        const long long v0 = crp[mo[i]];
        for (int64_t q = first; q < hi; q += 256) {
            const long long v = rp[q] - v0;
            if (rp64)
                ((long long *)out)[q] = v;
            else
                ((int *)out)[q] = (int)v;
        }
    });
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i <= count; i += (int64_t)gridDim.x * 256)
        bases[i] = crp[mo[i]];
}

static unsigned stack_grid(int64_t n)
{
    const int64_t chunks = (n + STACK_CHUNK - 1) / STACK_CHUNK;
    return (unsigned)(chunks < 1 ? 1 : chunks < 16384 ? chunks : 16384);
}

static unsigned grid_for(int64_t n)
{
    int64_t blocks = (n + 255) / 256;
    if (blocks > 16384)
        blocks = 16384;
    return (unsigned)(blocks < 1 ? 1 : blocks);
}

hipError_t launch_batch_rowptr(int which, int64_t count, const BatchInst *inst, BatchOffsets off, int64_t nrows,
                               int64_t nnz, int *out, DevStats *st, hipStream_t s)
{
    hipLaunchKernelGGL(k_batch_rowptr, dim3(stack_grid(nrows)), dim3(256), 0, s, which, (int)count, inst,
                       which ? off.ko : off.mo, which ? off.eb : off.ea, nrows, nnz, out, st);
    return hipGetLastError();
}

hipError_t launch_batch_entries(int which, int64_t count, const BatchInst *inst, BatchOffsets off, int64_t nnz,
                                int val32, int *Acol, int *Bcol, void *val, DevStats *st, hipStream_t s)
{
    if (nnz <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_batch_entries, dim3(stack_grid(nnz)), dim3(256), 0, s, which, (int)count, inst,
                       which ? off.eb : off.ea, off.ko, nnz, val32, Acol, Bcol, val, st);
    return hipGetLastError();
}

hipError_t launch_batch_split(int64_t count, BatchOffsets off, const long long *crp, void *out, int rp64,
                              long long *bases, int64_t nout, hipStream_t s)
{
    hipLaunchKernelGGL(k_batch_split, dim3(stack_grid(nout)), dim3(256), 0, s, (int)count, off.mo, crp, out, rp64,
                       bases);
    return hipGetLastError();
}

// ---- replayed plans --------------------------------------------------------------------------

__global__ void k_plan_check(DevStats *st, const DevStats *expect, int stage)
{
    if (threadIdx.x != 0 || blockIdx.x != 0)
        return;
    const BinStats &a = stage == 0 ? st->sym : st->num;
    const BinStats &b = stage == 0 ? expect->sym : expect->num;
    bool same = true;
    for (int k = 0; k < NBINS; ++k)
        same = same && a.count[k] == b.count[k] && a.max_need[k] == b.max_need[k] && a.max_span[k] == b.max_span[k] &&
               a.nsparse[k] == b.nsparse[k] && a.max_na[k] == b.max_na[k];
    if (stage == 0)
        same = same && st->dir_total == expect->dir_total && st->ntiles_b == expect->ntiles_b;
    else
        same = same && st->nnz_c == expect->nnz_c && st->wide_items == expect->wide_items &&
               st->hot_items == expect->hot_items;
    if (!same)
        st->err |= ERR_PLAN;
    if (st->err) {
        BinStats &w = stage == 0 ? st->sym : st->num;
        for (int k = 0; k < NBINS; ++k)
            w.count[k] = 0;
    }
}

hipError_t launch_plan_check(DevStats *st, const DevStats *expect, int stage, hipStream_t s)
{
    hipLaunchKernelGGL(k_plan_check, dim3(1), dim3(64), 0, s, st, expect, stage);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_plan_bases(const long long *__restrict__ got, const long long *__restrict__ want,
                                                    int64_t n, DevStats *st)
{
    bool diff = false;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        diff = diff || got[i] != want[i];
    if (diff)
        atomicOr(&st->err, ERR_PLAN);
}

hipError_t launch_plan_bases(const long long *got, const long long *want, int64_t n, DevStats *st, hipStream_t s)
{
    hipLaunchKernelGGL(k_plan_bases, dim3(grid_for(n)), dim3(256), 0, s, got, want, n, st);
    return hipGetLastError();
}

} // namespace hsmu
