// hsmu_internal.h -- declarations shared by the kernels (kernels.hip) and the host
// orchestrator (api.cpp).  Not part of the public ABI.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <mutex>

#include <hip/hip_runtime_api.h>

namespace hsmu {

// Row bins.  Bins 0..7 keep a row in LDS with G = 8 << b lanes per row (rows per
// workgroup = max(1, BLOCK / G)).  BIN_GLOBAL holds the rows that LDS does not, or not well: their
// directory is in global memory, and the numeric phase takes them in windows of C's columns.
constexpr int NLDS = 8;
constexpr int BIN_GLOBAL = 8;
constexpr int NBINS = 10; // as the public statistics (slot 9 stays empty)
// Workgroup size of the bins that pack several rows per workgroup (G < 64 lanes per
// row): one wave, so the phases of a row group are separated by single-wave barriers and
// every wave runs at its own pace (measured: 4-wave workgroups of 8-lane rows spend most
// of their time waiting at barriers for the slowest wave).
constexpr int BLOCK = 64;

// error bits raised on the device, reported at the next host synchronisation
constexpr int ERR_ROWPTR = 1;   // row pointer decreasing or out of [0, nnz]
constexpr int ERR_ACOL = 2;     // column of A outside [0, rows of B)
constexpr int ERR_BCOL = 4;     // column of B outside [0, N)
constexpr int ERR_UNSORTED = 8; // row of B with decreasing columns
constexpr int ERR_INTERNAL = 16;// symbolic and numeric counts disagree (a bug)
constexpr int ERR_PLAN = 32;    // a replayed plan's inputs changed structure

struct BinParams {
    int lds_block_budget; // LDS bytes per workgroup for bins with several rows per workgroup
    int lds_pair_budget;  // the same for two rows per workgroup
    int lds_row_max;      // LDS bytes one row may use
    int lds_window_max;   // the same for a row whose windows would be filled (window_filled)
    long long giant_min;  // products of a row that is wide whatever LDS it needs (wide_hot)
    int per_lane;         // work items per lane
    int lds_cu;           // LDS bytes of a CU
    int force_global;
    int min_waves;              // waves per CU a one-row workgroup's width should reach
};

struct BinStats {
    int count[NBINS];
    int max_need[NBINS]; // LDS bytes of the largest row in the bin
    int max_span[NBINS]; // tiles spanned by the widest row in the bin
    unsigned long long work[NBINS]; // products (numeric) or tile-products (symbolic)
    unsigned long long nnz_c[NBINS];// nnz of C in the bin's rows (symbolic: their products)
    unsigned long long nnz_a[NBINS];// nnz of A in the bin's rows
    int nsparse[NBINS];             // rows with a two-level tile directory
    int max_na[NBINS];              // longest row of A in the bin
};

// XCDs (accelerator complex dies, each with its own L2) the kernels map work onto: the
// device's count (hipDeviceAttributeNumberOfXccs; 8 on an MI355X, fewer in partitioned
// modes), at most this many.
constexpr int MAX_XCDS = 8;

// Device-side counters of one call, copied to pinned host memory at the two
// synchronisation points.
struct DevStats {
    unsigned long long dir_total; // directory entries reserved for rows in LDS bins
    long long nnz_c;
    int err;
    int ntiles_b;
    int pad;
    unsigned long long prod_most;     // products of the largest row, if more than WIDE_GIANT
    unsigned long long num_wide_work; // products of rows that may be wide in the numeric phase (symbolic binning)
    unsigned long long wide_items; // windows the wide rows may need, at most (numeric binning)
    unsigned long long hot_items;  // those of them that belong to hot rows
    unsigned long long hot_most;   // products beyond its entries of C of the hottest
    BinStats sym;
    BinStats num;
};

// The counters as a binning hands them to the host (pinned memory): seq, a number of the
// caller's, follows them.
struct HostStats {
    DevStats st;
    unsigned seq;
};

// A part of a binning's sums and maxima, for one bin: block b of the binning adds to part
// b % BIN_PARTS.
struct BinSum {
    unsigned long long work, nnz_c, nnz_a;
    unsigned need, span, na_max, nsparse;
};
constexpr int BIN_PARTS = 16;

// Work-queue counters of a persistent LDS kernel, one per XCD, each on a cache line of its own
// (on one line the pulls of all XCDs wait for each other: 200,000 rows of 8 entries times 24
// into 64 columns, 100,000 groups in each phase, 6.3 ms, so 1.6; 24 times 24 into 100,000
// columns 5.2 and 2.7).
constexpr int QUEUE_STRIDE = 32;
constexpr int QUEUE_INTS = MAX_XCDS * QUEUE_STRIDE;

// Everything on the device that a call needs zeroed: the counters, those of the work queues
// [phase][bin], the blocks done and the places taken of each binning or scan, and (behind it)
// the words of the two chained scans.
struct DevWork {
    DevStats st;
    alignas(128) unsigned queue[2][NBINS][QUEUE_INTS];
    BinSum sums[2][BIN_PARTS * NBINS]; // symbolic, numeric
    unsigned done[2], ticket[2];
    // followed by btiles_blocks(nnz(B)) + rowptr_blocks(M) 64-bit words
};

// Batched form: instance i of a batch, as seen by the stacking kernels.  The stacked A
// holds A_i's rows at mo.. and its entries at ea.., with columns shifted by ko (the first
// row of B_i in the stacked B); the stacked B holds B_i's rows at ko.. and entries at
// eb.., columns unchanged (so rows of the stacked C are the rows of C_i, columns local).
struct BatchInst {
    const int *Arp, *Acol;
    const void *Aval;
    const int *Brp, *Bcol;
    const void *Bval;
    int M, K, N, pad;
};

// Offsets of the instances, each array count+1 long (the last entry is the total):
// rows of A (mo), rows of B (ko), entries of A (ea), entries of B (eb).
struct BatchOffsets {
    const long long *mo, *ko, *ea, *eb;
};

#if defined(__HIPCC__)
#define HSMU_HD __host__ __device__
#else
#define HSMU_HD
#endif

// Accumulator form of a row in the numeric LDS kernel.  Compact (the HSMU form): exactly
// nnz(C_i) slots, column c in slot doff[t] + popcount(dm[t] & below(c & 63)).  Dense:
// one slot per column of the row's span, column c in slot c - 64*rmin, used when the
// span is at least two-thirds full (then the dense array costs at most 1.5x the compact
// one and saves the two directory reads per product) and at most 128 tiles wide.
HSMU_HD inline bool use_dense(int S, int n) { return S <= 128 && 2 * 64 * S <= 3 * n; }

// Tile directory of a row of C over its span [rmin, rmax] of S tiles.
// Flat: one entry (mask, first slot) per tile of the span, tile t at index t.
// Two-level, for rows whose span is mostly empty (the 3D stencil's A^2 row touches ~10 of
// ~140 tiles): a coarse bitmap of W = ceil(S/64) words marks the non-empty tiles, with
// coff[w] the compact index of the first non-empty tile of word w; the fine level holds
// only the non-empty tiles, tile t at compact index coff[t>>6] + popcount(cm[t>>6] &
// below(t&63)) -- the HSMU rank trick applied to tiles as well as to columns, so a slot
// is still found in O(1).  At most R = min(S, tile-products) fine entries.  Chosen when
// it at least halves the directory (never for spans of up to 64 tiles).
// (S is at most 2^25, so 32 bits hold all of this.)
HSMU_HD inline int fine_cap(int S, int tp) { return tp < S ? tp : S; }
HSMU_HD inline bool use_sparse(int S, int tp) { return S > 64 && 2 * (((S + 63) >> 6) + fine_cap(S, tp)) <= S; }
// directory entries of a row (12 bytes each when kept between the phases)
HSMU_HD inline int dir_entries(int S, int tp) { return use_sparse(S, tp) ? ((S + 63) >> 6) + fine_cap(S, tp) : S; }

// Sizes a row in LDS cannot have: layouts of larger rows are not worked out (32 bits) but
// given this many bytes.
constexpr int LAYOUT_CAP = 1 << 18;
constexpr int LAYOUT_NONE = 1 << 30;

// Tiles a row that shares a wave may span (its top words alone would fill a workgroup's LDS).
constexpr int SMALL_SPAN = 1 << 22;

// A B row with at least this many elements left in a window is walked by a whole wave (rows
// wider than LDS without an index of B).
constexpr int LONG_SEG = 256;

// ---- rows that share a wave ------------------------------------------------------------------
//
// G = 8, 16 or 32 lanes per row, each with SMALL_U pairs of elements of its B rows (a pair
// of an entry's odd last element is half empty) and one entry of A (32 lanes: or more):
//   rec    16[nA]   entries with elements: first less STREAM_V times the first pair, end, a_ij
//   ends   u32[U]   a bit per pair of each step of G: it ends an entry
//   top    8[...]   per 32 coarse words: which are marked, those before
//   coarse 8[...]   per 32 words (of 32 columns): which are marked, those before
//   fine   8[F]     per word: its columns, slots before
//   vals   f64[n]   numeric: accumulators
//   cols   i32[n]   numeric: columns
// (from ends to vals zeroed together, 16 bytes at a time; levels in fours)
// The fine level holds the marked words, at most one per product; with a word or less per
// product in the span it holds them all, and no level above it is needed (where all lanes
// would mark the same few bits).  The coarse level holds the span's coarse words, or, for a
// span of more than SMALL_DIRECT of them that the row leaves mostly empty, the marked ones.
constexpr int SMALL_U = 4;
constexpr int SMALL_DIRECT = 128;
struct SmallLayout {
    int rec, ends, top, coarse, fine, vals, cols, ntop, ncoarse, bytes;
    bool flat;
};
HSMU_HD inline int small_coarse(int S) { return (2 * S + 31) >> 5; }
HSMU_HD inline SmallLayout small_layout(bool numeric, bool tops, int S, int n, int nA, int p)
{
    SmallLayout L = {};
    const int words = 2 * S;
    L.flat = words <= p;
    const int f = L.flat ? words : p;
    int nc = L.flat ? 0 : small_coarse(S);
    if (tops && nc > SMALL_DIRECT && nc > 2 * (((nc + 31) >> 5) + p)) {
        L.ntop = (nc + 31) >> 5;
        nc = p;
    }
    L.ncoarse = nc;
    int o = 0;
    L.rec = o;
    o += 16 * nA;
    L.ends = o;
    o += 4 * SMALL_U;
    L.top = o;
    o += 8 * ((L.ntop + 3) & ~3);
    L.coarse = o;
    o += 8 * ((nc + 3) & ~3);
    L.fine = o;
    o += 8 * ((f + 3) & ~3);
    L.vals = o;
    if (numeric)
        o += 8 * n;
    L.cols = o;
    if (numeric)
        o += 4 * n;
    L.bytes = (o + 15) & ~15;
    return L;
}
// LDS of such a row on G lanes, if it is one: all its pairs fit
HSMU_HD inline int small_need(bool numeric, int G, int S, int n, int nA, long long p)
{
    return (nA <= G || G == 32) && p + nA <= 2 * SMALL_U * G && S <= SMALL_SPAN
               ? small_layout(numeric, true, S, n, nA, (int)p).bytes
               : LAYOUT_NONE;
}

// ---- one row per workgroup (64 lanes or more): the element stream ------------------------
//
// The B rows of a row's A entries are walked as one stream of slots of STREAM_V consecutive
// elements: entry e owns ceil(nnz(B_j) / STREAM_V) slots, and step s of the stream gives
// lane i of a wave slot 64 s + i, so every lane works whatever the lengths of the B rows,
// and each lane's elements come in one load.  (A load instruction costs a CU's L1 8.7
// cycles for 4 bytes per lane, 17.6 for 8 and 22 for 16, however few of its lanes are
// active: 29 bytes per cycle for full narrow loads, 46 for 16-byte ones.)  Up to G entries
// at a time are staged in LDS (start, end, a_ij: 16 bytes each), with a bit per slot that
// ends an entry and, per 64 slots, the entry of the first: a lane's entry is that number
// plus the bits below its slot.
constexpr int STREAM_V = 2;
// slots whose bits are in LDS at a time, for a row with G lanes
HSMU_HD constexpr int stream_window(int G) { return G * 32 > 4096 ? G * 32 : 4096; }

// LDS of one row (byte offsets), for a row of C over S tiles with n entries, nA entries in
// A, tp tile-products and p products:
//   vals f64[n]     accumulators (64*S of them in the dense form)
//   dm   u64[E]     tile masks (flat), or coarse words then fine masks (two-level)
//   rec  16[...]    staged entries: first element less STREAM_V times the first slot, end,
//                   a_ij; min(nA, G) of them
//   bits u64[...]   a bit per slot of the window: it ends an entry
//   doff u32[E]     slot of each tile's first column, coarse offsets (two-level)
//   ft   u32[R]     two-level: tile of each fine entry, relative to rmin
//   wb   u16[...]   entry of the first slot of each 64
struct StreamLayout {
    int vals, dm, rec, bits, doff, ft, wb, bytes;
};
HSMU_HD inline StreamLayout stream_layout(int G, int S, int n, int nA, int tp, long long p)
{
    StreamLayout L = {};
    const bool sparse = use_sparse(S, tp);
    const int E = dir_entries(S, tp);
    if (E > LAYOUT_CAP || n > LAYOUT_CAP) {
        L.bytes = LAYOUT_NONE;
        return L;
    }
    const long long slots = (p + (long long)nA * (STREAM_V - 1)) / STREAM_V;
    const int words = ((slots < stream_window(G) ? (int)slots : stream_window(G)) + 63) >> 6;
    int o = 8 * (!sparse && use_dense(S, n) ? 64 * S : n);
    o = (o + 15) & ~15;
    L.dm = o;
    o += 8 * E;
    o = (o + 15) & ~15;
    L.rec = o;
    o += 16 * (nA < G ? nA : G);
    L.bits = o;
    o += 8 * words;
    L.doff = o;
    o += 4 * E;
    L.ft = o;
    if (sparse)
        o += 4 * fine_cap(S, tp);
    L.wb = o;
    o += 2 * words;
    L.bytes = (o + 15) & ~15;
    return L;
}

// The symbolic counterpart: the stream is of tile pairs.
//   dm   u64[E]     tile masks (flat), or coarse words then fine masks (two-level)
//   rec, bits       as above
//   doff u32[E]     two-level: coarse offsets
//   wb   u16[...]   as above
HSMU_HD inline StreamLayout sym_stream_layout(int G, int S, int nA, int tp)
{
    StreamLayout L = {};
    const int E = dir_entries(S, tp);
    if (E > LAYOUT_CAP) {
        L.bytes = LAYOUT_NONE;
        return L;
    }
    const long long slots = ((long long)tp + (long long)nA * (STREAM_V - 1)) / STREAM_V;
    const int words = ((slots < stream_window(G) ? (int)slots : stream_window(G)) + 63) >> 6;
    int o = (8 * E + 15) & ~15;
    L.rec = o;
    o += 16 * (nA < G ? nA : G);
    L.bits = o;
    o += 8 * words;
    L.doff = o;
    if (use_sparse(S, tp))
        o += 4 * E;
    L.wb = o;
    o += 2 * words;
    L.bytes = (o + 15) & ~15;
    return L;
}

constexpr int BIN_SHARED = 3; // bins of rows that share a wave: 8, 16, 32 lanes

// Entries of A from which a row of few tiles per entry takes k_symbolic_wide: the stream's turns of
// 1,024 entries are a chain, its sub-groups of lanes are not (a row of
// 100,000 entries of 2 tiles 455 us as a stream, 235 so; 100 such rows, whole calls, 2.58 and 2.37 ms).
constexpr int SYM_LONG = 32 * 1024;
// LDS a row with p products needs in symbolic bin `bin`
HSMU_HD inline int sym_need(int bin, int S, int nA, int tp, long long p)
{
    if (nA >= SYM_LONG && tp / 4 <= nA)
        return LAYOUT_NONE;
    return bin >= BIN_SHARED ? sym_stream_layout(8 << bin, S, nA, tp).bytes : small_need(false, 8 << bin, S, 0, nA, p);
}

// ... and in numeric bin `bin`
HSMU_HD inline int num_need(int bin, int S, int n, int nA, int tp, long long p)
{
    return bin >= BIN_SHARED ? stream_layout(8 << bin, S, n, nA, tp, p).bytes : small_need(true, 8 << bin, S, n, nA, p);
}

// LDS kept back from the dynamic allocation for the kernels' static __shared__ arrays
constexpr int LDS_STATIC_RESERVE = 256;

// ---- launchers (kernels.hip); all enqueue on `s` and return the launch status ----

hipError_t launch_fill_zero(void *p, size_t bytes, hipStream_t s);

// One row of B as the row analysis needs it: entries, tiles (-1: see the tile pointers), first
// and last tile column (last = -1 for an empty row).
struct alignas(16) BRow {
    int len, ntiles, first, last;
};
// The records alone (and the number of tiles), for a B whose tiles may not be wanted.
hipError_t launch_brows(int64_t K, int64_t N, int64_t nnz, const int *rp, const int *col, BRow *brow, DevStats *st,
                        int num_cus, hipStream_t s);
// B -> tiles: tptr (K + 1), tcol and tmask (room for nnz), brow (K, may be null).  words:
// btiles_blocks(nnz) zeroed words, *ticket = 0.
int64_t btiles_blocks(int64_t nnz);
hipError_t launch_btiles(int64_t K, int64_t N, int64_t nnz, const int *rp, const int *col, int *tptr,
                         int *tcol, unsigned long long *tmask, BRow *brow, unsigned long long *words,
                         unsigned *ticket, DevStats *st, hipStream_t s);

// Per row of A: products, tile-products, tile span (from the BRow of each B_j it names), and
// the rows' symbolic bins: binrows, and each LDS-bin row's directory range: rdir[i] = offset
// (span entries), -1 for rows not in an LDS bin; st->dir_total = entries reserved.  host (may
// be null): the counters are copied there at the end (device-accessible host memory).
hipError_t launch_row_info(int64_t M, int64_t K, int64_t nnzA, const int *Arp, const int *Acol,
                           const BRow *brow, const int *tptr, long long *rprod, int *rtp, int *rmin,
                           int *rmax, int *rnnz, BinParams bp, int *binrows, long long *rdir, DevStats *st,
                           BinSum *sums, unsigned *done, HostStats *host, unsigned seq, int num_cus, hipStream_t s);

// C's row pointers (crp, and out32 when given: M + 1 each) from rnnz, and the numeric bins.
// words: rowptr_blocks(M) zeroed words, *ticket = 0.  sums, host as above (rowptr_blocks).
int64_t rowptr_blocks(int64_t M);
hipError_t launch_rowptr_bin(int64_t M, const int *Arp, const long long *rprod, const int *rtp,
                             const int *rmin, const int *rmax, const int *rnnz, long long *crp,
                             int *out32, BinParams bp, int *binrows, unsigned long long *words,
                             unsigned *ticket, DevStats *st, BinSum *sums, unsigned *done,
                             HostStats *host, unsigned seq, hipStream_t s);

// A kept directory that is two-level has this bit in rdir (the form follows from use_sparse
// for rows the symbolic phase held in LDS; it keeps flat ones for the others).
constexpr long long RDIR_TWO = 1LL << 62;

struct Operands {
    const int *Arp, *Acol;
    const void *Aval; // double, or float when val32
    const int *Brp, *Bcol;
    const void *Bval;
    int nnzB;  // >= STREAM_V (the host pads a smaller B)
    int val32;
    const int *tptr, *tcol;
    const unsigned long long *tmask;
    const int *rmin, *rmax;
    const int *rtp; // tile-products per row (chooses the directory form)
    const long long *rprod; // products per row
    // Row directories kept between the phases (nullptr when not kept): the symbolic LDS
    // kernel stores row i's directory (flat: tile masks and slot offsets; two-level: the
    // coarse words and compact indices, then the fine masks and slot offsets) at
    // dir_mask/dir_off + rdir[i]
    // (rdir < 0: not stored), the numeric kernel loads them instead of rebuilding them.
    const long long *rdir;
    unsigned long long *dir_mask;
    unsigned *dir_off;
};

// Rows that share a wave, those of the bins with count[b] > 0 in one launch (bin b's list at
// rows + b * stride, its needs and spans in bins).  Symbolic: rnnz; numeric: the rows of C,
// lds_bytes as launch_numeric.
enum { SMALL_SYMBOLIC, SMALL_F64, SMALL_F32C };
hipError_t launch_small(int form, const int *rows, long long stride, const BinStats *bins_dev, const int *count,
                        const BinStats &bins, const Operands &op, int *rnnz, const long long *crp, int *Ccol, void *Cval,
                        int *err, int num_cus, unsigned (*queue)[QUEUE_INTS], unsigned long long *lds_bytes, hipStream_t s);

// Global-memory workspace (bin BIN_GLOBAL): gws_blocks regions of gws_stride u64 each;
// a region holds gws_tiles 64-bit masks followed by gws_tiles 32-bit offsets, with
// gws_tiles >= the widest tile span in the bin.
// queue: nullptr = one workgroup per row group (grid from count); otherwise 8 zeroed
// counters and the LDS kernels run persistent (grid from occupancy x num_cus).
// two_level: some row of the bin has a two-level directory (BinStats::nsparse > 0).
// lds_dyn: LDS a row may use (lds_row_max); BIN_GLOBAL rows keep their flat directory in
// LDS when gws_stride masks fit it (gws is then unused).
hipError_t launch_symbolic(int bin, const int *rows, const int *count_dev, int count,
                           int max_need, int max_na, const Operands &op, int *rnnz, int tshift, int two_level,
                           unsigned long long *gws, long long gws_stride, int num_cus,
                           int gws_blocks, int lds_dyn, unsigned *queue, hipStream_t s);

// Wide rows (BIN_GLOBAL) in the numeric phase.  With kept directories and room for the index
// (below) they are processed as windows: a window is a run of units of WIDE_UNIT columns
// (aligned, so that all rows' windows share their boundaries) that holds at most WIDE_UNIT
// entries of C_i and spans at most WIDE_UMAX units, one workgroup each.  The index gives
// every B row's first element at each unit's start, so a window's elements are known without
// a search; where it does not pay, a window searches the B rows it names.
constexpr int WIDE_UNIT = 4096;
// Rows of more LDS than this are wide where the index pays: with one or two workgroups
// per CU they are slower in one piece.  R-MAT squares of scale 16 (FP32) / 18 with rows of up
// to 160 KB in LDS 2.35 / 17.1 ms, 80 KB 2.34 / 16.9, 64 KB 2.11 / 16.5, 48 KB 2.11 / 16.7.
constexpr int WINDOW_ROW_MIN = 64 * 1024;
// (the masks and slots of 24 units leave room for three workgroups per CU; R-MAT scale 18 with 4 /
// 8 / 16 / 24 units 17.8 / 17.8 / 16.4 / 16.2 ms, 4 and 8 in an earlier state that took 17.4 with 16)
constexpr int WIDE_UMAX = 24;
// The index costs a place per row of B and unit (2 to 3.4 ps each), whatever the wide rows are.
// A search costs a chain of loads per WIDE_STEP entries of A in a window, as long as a row of B
// takes halvings; with few entries in B's rows (up to two halvings) it costs what the index's two
// reads do.  The line lies between the products on both sides of it: rows of R-MAT scale 20 take
// with the index and without 3.8 and 4.1 ms (4 rows, 1,070 places per halving), 4.2 and 5.0 (16
// rows, 590), 8.9 and 14.3 (1,024 rows); rows of a Zipf panel 257 and 221 us (2 rows), 307 and 299
// (16 rows, 400), 420 and 426 (64 rows, 100), 4.14 and 5.38 ms (2,000 rows); R-MAT squares of
// scale 16 / 18 2.06 / 16.2 and 2.60 / 20.7 ms; a grid of 1 M rows, one of them with 20,000
// entries, 1.47 and 0.81 ms, of 4 M rows 13.7 (and 15 GB) and 4.6 ms; 200 rows of 50,000 entries
// times single ones 4.9 and 3.0 ms.
constexpr unsigned long long WIDE_INDEX_PLACES = 700;
constexpr int WIDE_STEP = 256;
constexpr int WIDE_TILES = WIDE_UNIT / 64;     // tiles of a unit
constexpr int WIDE_BUCKETS = 32;               // windows are listed by their place in C's columns
constexpr int WIDE_LISTS = 1 + 2 * WIDE_BUCKETS;
// Windows with a slot per column: of one unit, with at least WIDE_DENSE entries and fewer than
// WIDE_DENSE_WORK products (by the mean of their row), if there are WIDE_DENSE_MIN of them (a
// kernel of a few windows per workgroup is mostly its start and end).  They need neither
// masks nor slots per tile: a Zipf panel, whose windows hold 1.1 products per entry, takes
// 4.25 ms against 4.80.  Windows with more products are the hot columns of skewed graphs,
// where a slot per column puts more adds on one LDS bank: R-MAT squares of scale 16 and 18
// take 2.62 and 17.7 ms with them against 2.53 and 17.45.  Without the least number, scale 16 takes
// 2.03 ms against 2.00; without the form, Zipf panels of 2,000 / 777 rows 4.72 / 1.83 against 4.17 /
// 1.53.
// Windows of more than WIDE_HEAVY products are listed first, so that none of them is the last
// one running (one window of 1.1 M products, late in C's columns, among 541 M: 3.5 ms against 4.45;
// R-MAT squares and Zipf panels take the same time without).
constexpr int WIDE_DENSE = WIDE_UNIT / 4;
constexpr int WIDE_DENSE_WORK = 3 * WIDE_UNIT;
constexpr unsigned WIDE_DENSE_MIN = 8192;
constexpr int WIDE_HEAVY = 16 * WIDE_UNIT;
// Entries enough to fill a quarter of the row's windows; spread out further, it runs faster in one
// piece as long as LDS holds it (2,000 rows of 6,400 entries over 2 M columns: 738 us as 20 windows
// of 320 entries each, 320 us in LDS; an eighth or half in place of a quarter: the R-MAT square of
// scale 18 takes 16.15 and 16.64 ms, with a quarter 16.16).
HSMU_HD inline bool window_filled(int n, int S)
{
    return 4LL * n * WIDE_TILES * WIDE_UMAX >= (long long)S * WIDE_UNIT;
}
struct __attribute__((aligned(16))) WideItem {
    int row;
    unsigned units;     // first unit | number of units << 24
    unsigned base, cnt; // the row's entries before the window, and in it
};
// The list: windows with compact slots, from `dense` on those with a slot per column, its
// end; how many of each form are taken.  Windows that may be hot, the windows that are cut, their
// parts.
struct WideCount {
    unsigned dense, listed, taken[2];
    unsigned hot, sums;
    unsigned long long parts;
};
// A hot row has WIDE_HOT products more than entries of C_i, and entries of A for as many on a
// window's entries of C_i (each takes one product of an entry of A at most, unless B's rows repeat
// columns): one of its windows may hold as many, which kept a workgroup busy long after the others
// had ended.  Such windows are estimated from WIDE_SAMPLE of the row's entries of A and, with
// WIDE_HOT products or more and twice a workgroup's share of all wide rows' (less is no tail: cutting
// it slows an R-MAT square of scale 18 by 1.6%), cut into WIDE_PARTS or more ranges of entries of A
// (or of WIDE_PART_NA entries, up to WIDE_NA_PARTS of them: a workgroup takes 3.8 us for 256 entries
// of few elements), whose FP64 sums meet in memory.  3,000 rows of B with 900 of their 1,000 entries in one unit: a row
// of C with all of them 2.12 ms whole and 0.37 cut, 64 such rows 3.97 and 0.59.
constexpr unsigned long long WIDE_HOT = 512 * 1024;
constexpr int WIDE_PARTS = 4;
constexpr int WIDE_PART_NA = 4096;
constexpr int WIDE_NA_PARTS = 256;
constexpr int WIDE_SAMPLE = 256;
HSMU_HD inline bool wide_hot(long long p, long long n, int nA)
{
    return p - n > (long long)WIDE_HOT && (long long)nA * WIDE_UNIT >= (long long)WIDE_HOT;
}
// A row of this many products, and of twice a CU's share of all products, that fits LDS is wide for
// its windows to be cut: alone on a CU it ends long after the others (a row of 300,000 entries times
// 3 over 1,000 columns 3.0 ms in LDS, 1.37 cut; 50 dense rows of 4.5 M products 1.32 and 0.53 ms).
constexpr unsigned long long WIDE_GIANT = WIDE_HOT;
struct __attribute__((aligned(16))) WidePart {
    int row;
    unsigned units, base, cnt; // as the window's
    int e0, e1;                // entries of A
    int sum, pad;              // its place among the cut windows
};
struct WideSum { // where a cut window's values go in C, how many
    long long at;
    long long cnt;
};
HSMU_HD inline long long wide_units(long long N) { return (N + WIDE_UNIT - 1) / WIDE_UNIT; }
// windows of a row of n entries over S tiles, at most: two neighbouring ones hold more than
// WIDE_UNIT entries or span more than WIDE_UMAX units
HSMU_HD inline long long wide_row_items(int n, int S)
{
    return 2LL * (n / WIDE_UNIT) + 2LL * (S / (WIDE_TILES * WIDE_UMAX)) + 4;
}

// Otherwise one workgroup per row (blocks workgroups), each with a workspace of 3 *
// cur_stride + ft_stride ints (cursors, ends and next columns of its row's A entries:
// cur_stride >= the longest row of A in the bin; tiles of the fine directory entries of a
// two-level row: ft_stride >= the widest span in the bin).
struct WideRows {
    int *ws;
    long long cur_stride, ft_stride;
    int blocks;
    int lds_cu; // LDS bytes of a CU
    // windows: their capacity and list, the place of each listing workgroup's windows per
    // bucket, and how many are listed and taken (null items: one workgroup per row)
    long long items_cap;
    WideItem *items;
    unsigned *places;
    WideCount *ctr;
    int *index; // K rows of nunits + 1, or null: search
    long long nunits;
    long long K;
    // hot rows (null hot: none): their windows' places in the list, parts, cut windows with
    // WIDE_UNIT sums each; capacities
    unsigned *hot;
    WidePart *parts;
    WideSum *sums;
    double *sum_val;
    long long hot_cap, part_cap, sum_cap;
    long long hot_min; // products of a window that is cut
};
// workgroups that list the windows of count rows
int wide_item_blocks(int count, int num_cus);
// bytes of the lists besides the windows, at most (with what alignment adds)
inline unsigned long long wide_list_bytes(int num_cus)
{
    return 4ull * WIDE_LISTS * wide_item_blocks(INT_MAX, num_cus) + 2048;
}
size_t wide_ws_ints(long long cur_stride, long long ft_stride, int blocks);

// Numeric phase of one bin.  fp32c = 0: FP64 values (Cval double); fp32c = 1: compensated
// FP32 (Cval float).  lds_bytes (may be null): += the dynamic LDS of an LDS-bin launch,
// workgroups x bytes per workgroup (the reference's "practical need",
// compressed_Cval.cuh:202-533); the wide-row kernels' persistent workgroups reuse their LDS
// window by window and are not counted.
hipError_t launch_numeric(int bin, int fp32c, const int *rows, const int *count_dev, int count,
                          int max_need, int max_na, const Operands &op, const long long *crp, int *Ccol,
                          void *Cval, int bshift, int two_level, const WideRows &wide, int *err, int num_cus,
                          unsigned *queue, unsigned long long *lds_bytes,
                          hipStream_t s);

// A B of fewer than STREAM_V entries (n of them, at least one), copied to arrays of
// STREAM_V entries whose last one repeats: the element stream loads STREAM_V at a time.
hipError_t launch_pad_b(const int *col, const void *val, int val32, int n, int *pcol, void *pval, hipStream_t s);

// int64 row pointers that fit int32, as int32
hipError_t launch_rowptr_narrow(const long long *in, int64_t n, int *out, hipStream_t s);
// out[i] = in[i] - in[0] for i < n (row pointers of a row panel, rebased to 0)
hipError_t launch_rowptr_rebase(const int *in, int64_t n, int *out, hipStream_t s);
// sum[i] and asum[i] = sum of the values / of their magnitudes in row i of a CSR matrix
hipError_t launch_row_sums(int64_t M, const void *rp, int rp64, const void *val, int val32, double *sum,
                           double *asum, hipStream_t s);

// ---- batched form (kernels.hip) ----
// Stacked row pointers of A (which = 0, nrows = total rows of A) or B (which = 1): entry g
// of instance i = e0_i + rp_i[g - r0_i], the last entry = total entries.  Raises
// ERR_ROWPTR when an instance's rp[0] != 0 or rp[rows] != its nnz.
hipError_t launch_batch_rowptr(int which, int64_t count, const BatchInst *inst, BatchOffsets off,
                               int64_t nrows, int64_t nnz, int *out, DevStats *st, hipStream_t s);
// Stacked columns and values of B (which = 1) or A (0): Acol + ko_i, Bcol unchanged; either
// array may be nullptr (a batch of A_i * A_i takes both from one pass).  Raises ERR_ACOL /
// ERR_BCOL for a column outside instance i's range (and writes 0).
hipError_t launch_batch_entries(int which, int64_t count, const BatchInst *inst, BatchOffsets off,
                                int64_t nnz, int val32, int *Acol, int *Bcol, void *val, DevStats *st,
                                hipStream_t s);
// Row pointers of every C_i from the stacked C's (crp, int64): instance i's M_i + 1 entries
// at out + mo_i + i, rebased to start at 0; out is int64 (rp64) or int32.  Also
// bases[i] = crp[mo_i] for i <= count (where C_i's entries start).  nout = rows + count.
hipError_t launch_batch_split(int64_t count, BatchOffsets off, const long long *crp, void *out,
                              int rp64, long long *bases, int64_t nout, hipStream_t s);

// Replayed plans: compare the device's DevStats of one checkpoint (stage 0: after the
// symbolic binning, stage 1: after the numeric binning) with the recorded one; on any
// difference, or an input error already raised, set ERR_PLAN / keep err and zero the
// bin counts of that stage so that no later kernel runs on sizes the plan did not
// provision.
hipError_t launch_plan_check(DevStats *st, const DevStats *expect, int stage, hipStream_t s);
// Replayed batch plans: ERR_PLAN when the start of any C_i moved (its nnz changed).
hipError_t launch_plan_bases(const long long *got, const long long *want, int64_t n, DevStats *st,
                             hipStream_t s);

hipError_t launch_copy(const void *src, void *dst, size_t bytes, int num_cus, hipStream_t s);

// ---- allocation-free entry point (noalloc.hip) ----
// Bytes of the file-scope device array that is hsmu_spgemm_noalloc's whole workspace.
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)256 << 20;
// Device address of that array on `device`, which must be the current device: looked up
// once per device (hipGetSymbolAddress), then cached.
hipError_t scratch_setup(int device, void **ptr);
// Held for the whole of an hsmu_spgemm_noalloc call: calls on one device share its array.
std::mutex &scratch_lock(int device);

// Opt every kernel in to the device's full LDS size and tell the row kernels the device's
// XCD count (1..MAX_XCDS); call once per device, with it current.
hipError_t configure_kernels(int lds_max, int num_xcds);

} // namespace hsmu
