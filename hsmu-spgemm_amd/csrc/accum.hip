// accum.hip -- symbolic and numeric row kernels of the HSMU SpGEMM path for gfx950.
//
// Symbolic: nnz(C_i) from the OR of B's 64-column tile masks over row i of A, into the
// row's tile directory in LDS (flat: one mask per tile of the row's span; two-level for
// sparse spans: a coarse bitmap of the non-empty tiles, then their masks), with
// ds_or_b64; a popcount and a group scan give nnz(C_i) and each tile's first slot
// (reference: compressed_tilePtr_symbolic.cuh and compressed_tileOR.cuh, two hash
// passes over tiles there; one pass and no hashing here).
//
// Numeric: the HSMU accumulator -- exactly nnz(C_i) slots in LDS, the slot of column c
// being off[t] + popcount(mask[t] & below(c & 63)) for c's directory entry t, i.e. c's
// rank among C's sorted columns found in O(1) (reference: binary search over the sorted
// column list, src/compressed/compressed_Cval.cuh:5-69 and src/small/numeric.cuh:233-253);
// a dense form (one slot per column of a short, full span) skips the directory.  The
// numeric kernels also write C's sorted columns, replacing the reference's rank-sort pass
// (compressed_Ccol_symbolic.cuh:4-63).
//
// Rows of few products share a wave and keep their elements in registers; rows with a
// workgroup to themselves walk all their B rows as one stream of pairs of elements
// (symbolic: of tiles).
// Rows whose slice does not fit LDS (wide rows) use the windowed kernels at the end of this
// file.

#include <hip/hip_runtime.h>

#include <climits>

#include <type_traits>

#include "device_common.h"
#include "hsmu_internal.h"

namespace hsmu {

// XCDs of the device the row kernels map their row groups onto (configure_kernels sets
// it per device; each device holds its own copy).
static __constant__ int c_nxcd = MAX_XCDS;

// The one error these kernels raise; err may be host memory, hence a store.
DEVI void raise_internal(int *err) { __hip_atomic_store(err, ERR_INTERNAL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }

constexpr int UNROLL = 4;

// Compact index of tile t (relative to rmin) in a two-level directory: the rank of t
// among the row's non-empty tiles.
DEVI unsigned fine_index(const u64 *cm, const unsigned *coff, int t)
{
    const int w = t >> 6;
    return coff[w] + (unsigned)__popcll(cm[w] & below(t & 63));
}

// Walks over the row's tile-products (every tile of every B_j of the row):
//   OR_FLAT    dm[t] |= mask                  flat directory
//   OR_COARSE  cm[t >> 6] |= bit (t & 63)     two-level, pass 1: which tiles are non-empty
//   OR_FINE    fm[fine_index(t)] |= mask      two-level, pass 2
enum { OR_FLAT, OR_COARSE, OR_FINE };

template <int MODE>
DEVI void or_put(u64 *dm, const unsigned *coff, u64 *fm, int tt, u64 m)
{
    if constexpr (MODE == OR_FLAT)
        atomicOr(&dm[tt], m);
    else if constexpr (MODE == OR_COARSE)
        atomicOr(&dm[tt >> 6], 1ull << (tt & 63));
    else
        atomicOr(&fm[fine_index(dm, coff, tt)], m);
}

// Tiles [tb, te) of one B row into a flat directory by a group of gw lanes (this lane the gl-th),
// U tiles per lane per step.
template <int U> DEVI void or_walk(const Operands &op, int tb, int te, int gw, int gl, u64 *dm, int mn)
{
    for (int t = tb + gl; t < te; t += U * gw) {
        int c[U];
        u64 m[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int tu = t + u * gw;
            c[u] = -1;
            m[u] = 0;
            if (tu < te) {
                c[u] = op.tcol[tu];
                m[u] = op.tmask[tu];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c[u] >= 0)
                or_put<OR_FLAT>(dm, nullptr, nullptr, c[u] - mn, m[u]);
    }
}

// Each lane scans a contiguous chunk [ta, tb) of the n directory entries; groups of 256
// lanes or more visit it from s = ta + l mod chunk, wrapping round to ta: with every lane
// starting at its chunk's first entry, a chunk of 16 entries would put all 64 lanes of a
// wave on one LDS bank pair.  Smaller groups have short chunks and walk them from ta
// (s = ta) in one loop.  pre: the group's exclusive prefix of the popcounts at ta; head:
// the popcounts of [ta, s); tot: the group total.  Every thread of the workgroup must
// call it (G > 64 synchronises the workgroup).
struct ChunkScan {
    int ta, tb, s;
    unsigned pre, head, tot;
};
template <int G>
DEVI ChunkScan scan_popcounts(const u64 *m, int n, unsigned *redu)
{
    ChunkScan c;
    const int l = threadIdx.x & (G - 1);
    const int chunk = (n + G - 1) / G;
    c.ta = l * chunk;
    c.tb = c.ta + chunk < n ? c.ta + chunk : n;
    unsigned tail = 0, head = 0;
    if constexpr (G >= 256) {
        c.s = chunk > 1 ? c.ta + l % chunk : c.ta;
        if (c.s > c.tb)
            c.s = c.tb;
        for (int t = c.s; t < c.tb; ++t)
            tail += (unsigned)__popcll(m[t]);
        for (int t = c.ta; t < c.s; ++t)
            head += (unsigned)__popcll(m[t]);
    } else {
        c.s = c.ta;
        for (int t = c.ta; t < c.tb; ++t)
            tail += (unsigned)__popcll(m[t]);
    }
    c.head = head;
    c.pre = group_excl_scan<G>(tail + head, redu, c.tot);
    return c;
}

// The exclusive prefix at every entry of the lane's chunk, out(t, prefix, m[t]), in the
// scan's visiting order.  Each entry is read before out is called for it, so out may
// overwrite m[t] itself.
template <int G, typename Out>
DEVI void chunk_offsets(const u64 *m, const ChunkScan &c, Out out)
{
    if constexpr (G >= 256) {
        unsigned p = c.pre + c.head;
        for (int t = c.s; t < c.tb; ++t) {
            const u64 w = m[t];
            out(t, p, w);
            p += (unsigned)__popcll(w);
        }
        p = c.pre;
        for (int t = c.ta; t < c.s; ++t) {
            const u64 w = m[t];
            out(t, p, w);
            p += (unsigned)__popcll(w);
        }
    } else {
        unsigned p = c.pre;
        for (int t = c.ta; t < c.tb; ++t) {
            const u64 w = m[t];
            out(t, p, w);
            p += (unsigned)__popcll(w);
        }
    }
}

// Where row's kept directory lies, -1 if it has none in the form the row takes here (a row
// the symbolic phase held in global memory keeps a flat one).
DEVI long long kept_dir(const Operands &op, int row, bool two)
{
    const long long rd = op.rdir[row];
    return rd >= 0 && ((rd & RDIR_TWO) != 0) == two ? rd & ~RDIR_TWO : -1;
}

// ---- numeric forms ---------------------------------------------------------------------
//
// A slot is one double in both forms, so the LDS layout, the bins and the adds
// (ds_add_f64) are the same.
// PrecF64 (plain): FP64 values.
// PrecF32C (compensated FP32): FP32 values.  The product of two FP32 values is exact in
// FP64 (24 + 24 bits), so a double slot takes the place of a (sum, compensation) pair of
// floats: it carries 53 bits where the pair carries 48, and one ds_add_f64 takes the place
// of a read, TwoProduct, TwoSum and a 64-bit compare-and-swap loop.  The sum is rounded to
// FP32 once, at the end.  One CU retires a wave's ds_add_f64 on random slots in 24 cycles;
// the compare-and-swap form measured 1.9 times the numeric time of this one on a banded
// matrix.
struct PrecF64 {
    typedef double V;
    static DEVI double prep(double a, V b) { return a * b; }
    static DEVI void put(double *vals, unsigned slot, double p) { atomicAdd(&vals[slot], p); }
    static DEVI void add(double *vals, unsigned slot, double a, V b) { put(vals, slot, prep(a, b)); }
    static DEVI V result(const double *vals, unsigned slot) { return vals[slot]; }
};

struct PrecF32C {
    typedef float V;
    static DEVI double prep(double a, V b) { return a * (double)b; }
    static DEVI void put(double *vals, unsigned slot, double p) { atomicAdd(&vals[slot], p); }
    static DEVI void add(double *vals, unsigned slot, double a, V b) { put(vals, slot, prep(a, b)); }
    static DEVI V result(const double *vals, unsigned slot) { return (float)vals[slot]; }
};

// Slot of column c in the row's accumulator, by directory form.
enum { SLOT_FLAT, SLOT_DENSE, SLOT_TWO_LEVEL };

// ---- the element stream of a row ------------------------------------------------------------
//
// One workgroup of G lanes (64 or more) walks the B rows of its row's A entries as one
// stream of slots (hsmu_internal.h).  stage() takes one entry per lane, mark() lays out the
// bits of a window of slots, run() goes over all of a row's entries: entry(e) gives entry
// e's first element, length and payload, body(st, w0) walks the window of slots from w0.
struct Segment {
    int start, len;
    u64 payload;
};

template <int G> struct Stream {
    static constexpr int NW = G / 64;
    static constexpr int WINDOW = stream_window(G);
    uint4 *rec;
    u64 *bits, *red;
    unsigned short *wb;
    long long first, total; // this lane's first slot, slots in all
    int cnt, nrec;          // this lane's slots, entries with slots
    unsigned rank;

    DEVI void stage(const Segment &g)
    {
        cnt = (int)(((unsigned)g.len + STREAM_V - 1) / STREAM_V);
        u64 tot;
        const u64 ex = group_excl_scan<G, u64>((u64)(unsigned)cnt | (cnt ? 1ull << 48 : 0ull), red, tot);
        first = (long long)(ex & ((1ull << 48) - 1));
        rank = (unsigned)(ex >> 48);
        total = (long long)uniform64(tot & ((1ull << 48) - 1));
        nrec = (int)uniform((unsigned)(tot >> 48));
        if (cnt)
            rec[rank] = make_uint4((unsigned)g.start - STREAM_V * (unsigned)first, (unsigned)(g.start + g.len),
                                   (unsigned)g.payload, (unsigned)(g.payload >> 32));
    }
    DEVI void mark(long long w0)
    {
        if (!cnt)
            return;
        const long long f = first - w0, last = f + cnt - 1;
        if (last >= 0 && last < WINDOW)
            atomicOr(&bits[last >> 6], 1ull << (last & 63));
        const int s0 = f > 0 ? (f < WINDOW ? (int)((f + 63) >> 6) : WINDOW / 64) : 0;
        const int s1 = last < 0 ? -1 : (last < WINDOW ? (int)(last >> 6) : WINDOW / 64 - 1);
        for (int s = s0; s <= s1; ++s)
            wb[s] = (unsigned short)rank;
    }
    // steps of 64 slots in the window from w0
    DEVI int steps(long long w0) const
    {
        const long long n = total - w0 < WINDOW ? total - w0 : WINDOW;
        return (int)((n + 63) >> 6);
    }
    // the entry of this lane's slot in step s of the window (past the last slot: any)
    DEVI uint4 entry(int s) const { return entry(wb[s], bits[s]); }
    DEVI uint4 entry(int base, u64 word) const
    {
        int e = base + mbcnt(word);
        e = e < nrec ? e : nrec - 1;
        return rec[e];
    }
    // The bits must be zero, and a barrier passed since.  col_of(e) loads entry e's column
    // and entry_of(e, col) the rest; past the row's end they give an empty entry.  Those of
    // the next G entries, and the columns of the G after them, are loaded while the body
    // walks these.
    template <typename Col, typename Entry, typename Body>
    DEVI void run(int nA, const Segment &s0, Col col_of, Entry entry_of, Body body)
    {
        const int l = threadIdx.x;
        Segment g = s0;
        int j = G < nA ? col_of(G + l) : 0;
        for (int c = 0; c < nA; c += G) {
            stage(g);
            if (c + G < nA) {
                g = entry_of(c + G + l, j);
                if (c + 2 * G < nA)
                    j = col_of(c + 2 * G + l);
            }
            for (long long w0 = 0; w0 < total; w0 += WINDOW) {
                mark(w0);
                __syncthreads();
                body(*this, w0);
                __syncthreads();
                if (c + G < nA || w0 + WINDOW < total) {
                    const int n = steps(w0);
                    for (int q = l; q < n; q += G)
                        bits[q] = 0;
                    __syncthreads();
                }
            }
        }
    }
    template <typename Entry, typename Body> DEVI void run(int nA, Entry entry_of, Body body)
    {
        const int l = threadIdx.x;
        for (int c = 0; c < nA; c += G) {
            stage(c + l < nA ? entry_of(c + l) : Segment{0, 0, 0});
            for (long long w0 = 0; w0 < total; w0 += WINDOW) {
                mark(w0);
                __syncthreads();
                body(*this, w0);
                __syncthreads();
                if (c + G < nA || w0 + WINDOW < total) {
                    const int n = steps(w0);
                    for (int q = l; q < n; q += G)
                        bits[q] = 0;
                    __syncthreads();
                }
            }
        }
    }
};

// STREAM_V consecutive elements in one load, at the alignment of a single element.
template <typename T> struct Vec2 {
    typedef T type __attribute__((ext_vector_type(2), aligned(sizeof(T))));
};
template <typename T> DEVI typename Vec2<T>::type load2(const T *p) { return *(const typename Vec2<T>::type *)p; }

// Entry e of a row of nA entries from a0: its column, and the tiles of that row of B (none past
// the row's end).
DEVI int col_of(const Operands &op, int a0, int e, int nA) { return e < nA ? op.Acol[a0 + e] : 0; }
DEVI Segment tile_range(const Operands &op, int e, int nA, int j)
{
    if (e >= nA)
        return Segment{0, 0, 0};
    const typename Vec2<int>::type t = load2(op.tptr + j);
    return Segment{t.x, t.y - t.x, 0};
}

// A lane's elements k, k + 1 of an array of n: loaded from k or, at the array's end, from
// n - 2; in0 / in1: element 0 / 1 of the load belongs to [k, end).
struct Pair {
    unsigned at;
    bool in0, in1;
    DEVI Pair(unsigned k, unsigned end, unsigned n)
    {
        at = k < n - 2 ? k : n - 2;
        in0 = at == k && k < end;
        in1 = at + 1 >= k && at + 1 < end;
    }
};

// Add the products of a window of the row's stream into their slots, STREAM_U steps of a
// wave loaded while the STREAM_U before them are added (the loads are not predicated, so
// that a wait for one set is not a wait for the other).
constexpr int STREAM_U = 2;
template <int G, int FORM, typename P, typename Off>
DEVI void stream_add(const Stream<G> &st, long long w0, const Operands &op, const u64 *cm, const unsigned *coff,
                     const u64 *fm, const Off *foff, double *vals, int mn)
{
    typedef typename P::V V;
    constexpr int NW = G / 64, U = STREAM_U;
    const V *__restrict__ Bval = (const V *)op.Bval;
    const unsigned nB = (unsigned)op.nnzB;
    const int c0 = mn << 6;
    const int lane = threadIdx.x & 63;
    const int nst = st.steps(w0);
    int s = NW > 1 ? uniform((int)(threadIdx.x >> 6)) : 0;
    if (s >= nst)
        return;
    typename Vec2<int>::type c[2][U];
    typename Vec2<V>::type v[2][U];
    double a[2][U];
    bool in0[2][U], in1[2][U];
    // lane i holds the bits and the first entry of the wave's i-th next step
    static_assert(Stream<G>::WINDOW / 64 <= 64 * NW, "a wave's steps fit its lanes");
    u64 lw = 0;
    int lb = 0;
    if (s + lane * NW < nst) {
        lw = st.bits[s + lane * NW];
        lb = st.wb[s + lane * NW];
    }
    int i = 0; // the wave's next step
    auto load = [&](int h) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // past the wave's last step: some entry, with nothing in it
            const uint4 r = st.entry(__builtin_amdgcn_readlane(lb, (i + u) & 63), readlane_u64(lw, (i + u) & 63));
            const int su = s + u * NW;
            const unsigned k = r.x + STREAM_V * ((unsigned)w0 + 64 * su + lane);
            const Pair q(k, su < nst ? r.y : 0u, nB);
            c[h][u] = load2(op.Bcol + q.at);
            v[h][u] = load2(Bval + q.at);
            a[h][u] = __longlong_as_double((long long)(((u64)r.w << 32) | r.z));
            in0[h][u] = q.in0;
            in1[h][u] = q.in1;
        }
        i += U;
        s += U * NW;
    };
    auto slot_of = [&](int col) -> unsigned {
        const int q = col - c0;
        if constexpr (FORM == SLOT_DENSE) {
            return (unsigned)q;
        } else {
            const unsigned kk = FORM == SLOT_TWO_LEVEL ? fine_index(cm, coff, q >> 6) : (unsigned)(q >> 6);
            return foff[kk] + (unsigned)__popcll(fm[kk] & below(q & 63));
        }
    };
    auto add = [&](int h) {
        unsigned s0[U], s1[U];
        double p0[U], p1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (FORM == SLOT_DENSE || in0[h][u])
                s0[u] = slot_of(c[h][u].x);
            if (FORM == SLOT_DENSE || in1[h][u])
                s1[u] = slot_of(c[h][u].y);
            p0[u] = P::prep(a[h][u], v[h][u].x);
            p1[u] = P::prep(a[h][u], v[h][u].y);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (in0[h][u])
                P::put(vals, s0[u], p0[u]);
            if (in1[h][u])
                P::put(vals, s1[u], p1[u]);
        }
    };
    load(0);
    while (true) {
        const bool m1 = s < nst;
        if (m1)
            load(1);
        add(0);
        if (!m1)
            break;
        const bool m0 = s < nst;
        if (m0)
            load(0);
        add(1);
        if (!m0)
            break;
    }
}

// OR a window of the row's tile stream (entries are tile ranges) into its directory, OR_U
// steps of a wave loaded together.
constexpr int OR_U = 4;
template <int G, int MODE>
DEVI void stream_or(const Stream<G> &st, long long w0, const Operands &op, u64 *dm, const unsigned *coff, u64 *fm, int mn)
{
    constexpr int NW = G / 64;
    const unsigned nB = (unsigned)op.nnzB;
    const int lane = threadIdx.x & 63;
    const int nst = st.steps(w0);
    const int s0 = NW > 1 ? uniform((int)(threadIdx.x >> 6)) : 0;
    u64 lw = 0; // lane i holds the wave's i-th step
    int lb = 0;
    if (s0 + lane * NW < nst) {
        lw = st.bits[s0 + lane * NW];
        lb = st.wb[s0 + lane * NW];
    }
    for (int i = 0, s = s0; s < nst; i += OR_U, s += OR_U * NW) {
        Vec2<int>::type c[OR_U];
        Vec2<u64>::type m[OR_U];
        bool in0[OR_U], in1[OR_U];
#pragma unroll
        for (int u = 0; u < OR_U; ++u) {
            const uint4 r = st.entry(__builtin_amdgcn_readlane(lb, (i + u) & 63), readlane_u64(lw, (i + u) & 63));
            const int su = s + u * NW;
            const Pair q(r.x + STREAM_V * ((unsigned)w0 + 64 * su + lane), su < nst ? r.y : 0u, nB);
            c[u] = load2(op.tcol + q.at);
            if constexpr (MODE != OR_COARSE)
                m[u] = load2(op.tmask + q.at);
            else
                m[u] = Vec2<u64>::type{0, 0};
            in0[u] = q.in0;
            in1[u] = q.in1;
        }
#pragma unroll
        for (int u = 0; u < OR_U; ++u) {
            if (in0[u])
                or_put<MODE>(dm, coff, fm, c[u].x - mn, m[u].x);
            if (in1[u])
                or_put<MODE>(dm, coff, fm, c[u].y - mn, m[u].y);
        }
    }
}

// ---- symbolic ------------------------------------------------------------------------------

// ---- rows that share a wave ----------------------------------------------------------------
//
// Rows of few products, G = 8, 16 or 32 lanes each (small_layout): the row's elements of B
// are loaded once, SMALL_U pairs per lane, and stay in registers.  Their columns mark the
// row's words (32 columns each) in a coarse bitmap; a scan gives the marked words compact
// places, where the columns are marked in turn; a second scan gives nnz(C_i) -- all the
// symbolic phase wants -- and each word's first slot.  (Narrow spans need no coarse level, wide
// ones have another above it: small_layout.)  The numeric phase then adds every
// product at its column's rank (ds_add_f64), puts the column there too, and the row goes
// out in order.
// Against staging the A entries in LDS and walking B's tiles twice for the directory and
// its rows a third time for the products, a lane or two per row of B (512 Laplacians of
// 7.5 M rows; that kernel spent 52% of its time in vector instructions, 62% in the L1 and
// 39% in LDS, two thirds of it bank conflicts): numeric 2,860 -> 1,670 us, symbolic 1,044
// -> 880 us, the call 5.74 -> 4.41 ms; a 47^3 stencil 178 -> 147 us, a random product of
// ragged rows 261 -> 197 us.  Now bound by vector instructions (about half of the time) and
// the chain of loads, row to entries to B.  5 waves per SIMD (102 registers): at 4 the
// batch's numeric phase takes 1,760 us, at 6 it spills (3,040 us).
struct SmallNone { // symbolic: no values
    typedef float V;
};
// TOPS: some row of the launch may have a third level (which costs registers).
template <int G, typename P, bool TOPS>
DEVI void small_rows(const int *__restrict__ rows, const int *__restrict__ count_p, int slice_bytes, const Operands &op,
                     int *__restrict__ rnnz, const long long *__restrict__ crp, int *__restrict__ Ccol,
                     typename P::V *__restrict__ Cval, int *err, unsigned *queue, int block, int blocks)
{
    typedef typename P::V V;
    constexpr bool NUM = !std::is_same<P, SmallNone>::value;
    constexpr int RPB = BLOCK / G, U = SMALL_U;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ int grp_s[2];
    const int g = threadIdx.x / G, l = threadIdx.x & (G - 1);
    unsigned char *slice = lds + (size_t)g * slice_bytes;
    const V *__restrict__ Aval = (const V *)op.Aval;
    const V *__restrict__ Bval = (const V *)op.Bval;
    const unsigned nB = (unsigned)op.nnzB;
    const int nrows = *count_p;
    // bits of a word below a column, or of a step's ends below a lane
    auto under = [](unsigned m, int c) { return m & ((1u << (c & 31)) - 1u); };
    for (GroupWalk gw(queue, (nrows + RPB - 1) / RPB, grp_s, c_nxcd, block, blocks); gw.more(); gw.next()) {
        const int idx = gw.grp * RPB + g;
        const int row = idx < nrows ? rows[idx] : -1;
        int S = 0, w0 = 0, n = 0, a0 = 0, nA = 0, p = 0;
        long long cb = 0;
        if (row >= 0) {
            w0 = 2 * op.rmin[row];
            S = op.rmax[row] - (w0 >> 1) + 1;
            a0 = op.Arp[row];
            nA = op.Arp[row + 1] - a0;
            p = (int)op.rprod[row];
            if constexpr (NUM) {
                cb = crp[row];
                n = (int)(crp[row + 1] - cb);
            }
        }
        const SmallLayout L = small_layout(NUM, TOPS, S, n, nA, p);
        uint2 *tops = (uint2 *)(slice + L.top);
        uint2 *coarse = (uint2 *)(slice + L.coarse); // words of the row: marked words, those before
        uint2 *fine = (uint2 *)(slice + L.fine);     // marked words: columns, slots before
        double *vals = (double *)(slice + L.vals);
        int *cols = (int *)(slice + L.cols);
        uint4 *rec = (uint4 *)(slice + L.rec);
        unsigned *ends = (unsigned *)(slice + L.ends); // per step of G pairs: it ends an entry
        // (the last 16 bytes may reach into cols, which is written later, or past the layout's
        // end, which is a multiple of 16)
        auto clear = [&]() {
            for (int q = L.ends + 16 * l; q < (NUM ? L.cols : L.vals); q += 16 * G)
                *(uint4 *)(slice + q) = make_uint4(0, 0, 0, 0);
        };
        // the entries of A, one per lane at a time: their pairs among the row's
        unsigned total = 0, nrec = 0;
        for (int c = 0; c == 0 || (G == 32 && __any(c < nA)); c += G) {
            int start = 0, len = 0;
            u64 a = 0;
            if (c + l < nA) {
                const typename Vec2<int>::type b = load2(op.Brp + op.Acol[a0 + c + l]);
                start = b.x;
                len = b.y - b.x;
                if constexpr (NUM)
                    a = (u64)__double_as_longlong((double)Aval[a0 + c + l]);
            }
            if (c == 0)
                clear();
            const unsigned cnt = (unsigned)(len + 1) >> 1;
            unsigned tot;
            const unsigned ex = group_excl_scan<G, unsigned>(cnt | (cnt ? 1u << 16 : 0u), nullptr, tot);
            const unsigned first = total + (ex & 0xffff);
            __syncthreads();
            if (cnt) {
                const unsigned last = first + cnt - 1;
                atomicOr(&ends[last / G], 1u << (last & (G - 1)));
                rec[nrec + (ex >> 16)] = make_uint4((unsigned)start - STREAM_V * first, (unsigned)(start + len),
                                                    (unsigned)a, (unsigned)(a >> 32));
            }
            total += tot & 0xffff;
            nrec += tot >> 16;
        }
        __syncthreads();
        // element 0 of a live pair is always the row's (at the array's end it is the load's
        // second), element 1 if the entry has it
        int c0[U], c1[U];
        V v0[U], v1[U];
        double av[U];
        bool live[U], two[U];
        unsigned e = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned bits = ends[u];
            const unsigned q = u * G + l;
            live[u] = q < total;
            two[u] = false;
            c0[u] = c1[u] = 0;
            if (live[u]) {
                const uint4 r = rec[e + __popc(under(bits, l))];
                const unsigned k = r.x + STREAM_V * q, at = k < nB - 2 ? k : nB - 2;
                const typename Vec2<int>::type c = load2(op.Bcol + at);
                c0[u] = at == k ? c.x : c.y;
                c1[u] = c.y;
                two[u] = k + 1 < r.y;
                if constexpr (NUM) {
                    const typename Vec2<V>::type v = load2(Bval + at);
                    v0[u] = at == k ? v.x : v.y;
                    v1[u] = v.y;
                    av[u] = __longlong_as_double((long long)(((u64)r.w << 32) | r.z));
                }
            }
            e += __popc(bits);
        }
        // exclusive prefix of the words' bits in their second halves, four words a lane; the sum
        auto prefix = [&](uint2 *m, int nw) {
            unsigned sum = 0;
            for (int q0 = 0; __any(q0 < nw); q0 += 4 * G) {
                const int q = q0 + 4 * l;
                uint4 a = make_uint4(0, 0, 0, 0), b = a;
                if (q < nw) {
                    a = *(uint4 *)(m + q);
                    b = *(uint4 *)(m + q + 2);
                }
                const unsigned k0 = __popc(a.x), k1 = k0 + __popc(a.z), k2 = k1 + __popc(b.x);
                unsigned t;
                const unsigned x = sum + group_excl_scan<G, unsigned>(k2 + __popc(b.z), nullptr, t);
                if (q < nw) {
                    *(uint4 *)(m + q) = make_uint4(a.x, x, a.z, x + k0);
                    *(uint4 *)(m + q + 2) = make_uint4(b.x, x + k1, b.z, x + k2);
                }
                sum += t;
            }
            return sum;
        };
        // a column's word, and its place in the coarse and fine level once those above are done
        auto word = [&](int c) { return (c >> 5) - w0; };
        auto place = [&](const uint2 *m, int w) {
            const uint2 x = m[w >> 5];
            return x.y + (unsigned)__popc(under(x.x, w));
        };
        auto coarse_of = [&](int w) { return TOPS && L.ntop ? place(tops, w >> 5) : (unsigned)w >> 5; };
        auto mark = [&](uint2 *m, unsigned at, int bit) { atomicOr(&m[at].x, 1u << (bit & 31)); };
        int nc = L.ncoarse;
        if constexpr (TOPS) {
            if (__any(L.ntop > 0)) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (live[u] && L.ntop)
                        mark(tops, (unsigned)word(c0[u]) >> 10, word(c0[u]) >> 5);
                    if (two[u] && L.ntop)
                        mark(tops, (unsigned)word(c1[u]) >> 10, word(c1[u]) >> 5);
                }
                __syncthreads();
                const int marked = (int)prefix(tops, L.ntop);
                nc = L.ntop ? marked : nc;
                __syncthreads();
            }
        }
        // mark the words
        int nf = 2 * S;
        if (__any(!L.flat)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (live[u] && !L.flat)
                    mark(coarse, coarse_of(word(c0[u])), word(c0[u]));
                if (two[u] && !L.flat)
                    mark(coarse, coarse_of(word(c1[u])), word(c1[u]));
            }
            __syncthreads();
            const int marked = (int)prefix(coarse, nc);
            nf = L.flat ? nf : marked;
            __syncthreads();
        }
        // mark the columns
        unsigned f0[U], f1[U];
        auto fine_of = [&](int c) {
            const int w = word(c);
            const uint2 x = coarse[coarse_of(w)]; // (a flat row's lies in its fine level)
            return L.flat ? (unsigned)w : x.y + (unsigned)__popc(under(x.x, w));
        };
#pragma unroll
        for (int u = 0; u < U; ++u) {
            f0[u] = f1[u] = 0;
            if (live[u]) {
                f0[u] = fine_of(c0[u]);
                mark(fine, f0[u], c0[u]);
            }
            if (two[u]) {
                f1[u] = fine_of(c1[u]);
                mark(fine, f1[u], c1[u]);
            }
        }
        __syncthreads();
        if constexpr (!NUM) {
            unsigned k = 0;
            for (int q = l; q < nf; q += G)
                k += __popc(fine[q].x);
            k = group_sum<G>(k);
            if (row >= 0 && l == 0)
                rnnz[row] = (int)k;
        } else {
            const bool ok = (int)prefix(fine, nf) == n;
            if (row >= 0 && !ok && l == 0)
                raise_internal(err);
            __syncthreads();
            if (ok) {
                auto put = [&](unsigned f, int c, double x) {
                    const uint2 m = fine[f];
                    const unsigned slot = m.y + (unsigned)__popc(under(m.x, c));
                    cols[slot] = c;
                    P::put(vals, slot, x);
                };
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (live[u])
                        put(f0[u], c0[u], P::prep(av[u], v0[u]));
                    if (two[u])
                        put(f1[u], c1[u], P::prep(av[u], v1[u]));
                }
            }
            __syncthreads();
            if (ok)
                for (int q = l; q < n; q += G) {
                    Ccol[cb + q] = cols[q];
                    Cval[cb + q] = P::result(vals, (unsigned)q);
                }
        }
        __syncthreads();
    }
}

// One bin of such rows; or, where several have rows, the three in one launch, those of the
// widest groups first (a launch of a few thousand rows is all start and end: a random product
// of 30,011 ragged rows takes 164 us in place of 199; but with the registers of the widest
// form a batch whose rows are all of one bin takes 3.79 ms in place of 3.70).  That launch gets 4
// waves per SIMD: at 5 it spills 34 registers (200,000 rows of 3 times 3 160 us, 154 at 4).
template <int G, typename P, bool TOPS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_small_bin(
    const int *__restrict__ rows, const int *__restrict__ count, int slice, Operands op, int *__restrict__ rnnz,
    const long long *__restrict__ crp, int *__restrict__ Ccol, typename P::V *__restrict__ Cval, int *err,
    unsigned *queue)
{
    small_rows<G, P, TOPS>(rows, count, slice, op, rnnz, crp, Ccol, Cval, err, queue, blockIdx.x, gridDim.x);
}

struct SmallBins {
    const int *rows[BIN_SHARED], *count[BIN_SHARED];
    unsigned *queue[BIN_SHARED];
    int slice[BIN_SHARED], blocks[BIN_SHARED];
};
template <typename P, bool TOPS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_small_rows(
    SmallBins bins, Operands op, int *__restrict__ rnnz, const long long *__restrict__ crp, int *__restrict__ Ccol,
    typename P::V *__restrict__ Cval, int *err)
{
    int block = blockIdx.x;
#define SMALL(B, G)                                                                                                    \
    if (block < bins.blocks[B])                                                                                        \
        return small_rows<G, P, TOPS>(bins.rows[B], bins.count[B], bins.slice[B], op, rnnz, crp, Ccol, Cval, err,      \
                                      bins.queue[B], block, bins.blocks[B]);                                           \
    block -= bins.blocks[B];
    SMALL(2, 32) SMALL(1, 16) SMALL(0, 8)
#undef SMALL
}

// nnz(C_i) for a row with a workgroup to itself: the tiles of its B rows, walked as one
// stream of pairs, are ORed into the row's tile directory (ds_or_b64), and its bits counted.
// Flat rows: one pass into a directory over the whole span.  Two-level rows: pass 1 marks
// the non-empty tiles in the coarse bitmap, a scan gives their compact indices, pass 2 ORs
// the masks into the compact fine level.  Bound by the loads of column and mask per tile (a load instruction costs
// the same for any number of active lanes: B rows of a few tiles left most of a sub-group
// idle, and staging entries in LDS doubled a row's need) and then by the LDS ORs.  Symbolic
// stage of R-MAT squares, before and after: scale 16 938 and 434 us, scale 18 8.5 and
// 3.5 ms; banded rows of 100 tiles 147 and 131 us.  TL: some row of the launch has a two-level directory.  A kept directory
// goes out coalesced: the masks first, then each entry's slot offset, written over its mask
// in LDS (coarse level: into doff, which the fine pass reads).
template <int G, bool TL, bool LONG = false>
__global__ __launch_bounds__(G) void k_symbolic_row(const int *__restrict__ rows, const int *__restrict__ count_p,
                                                    Operands op, int *__restrict__ rnnz, unsigned *queue)
{
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ u64 red[16];
    __shared__ int grp_s[2];
    const int l = threadIdx.x;
    const int nrows = *count_p;
    for (GroupWalk gw(queue, nrows, grp_s, c_nxcd); gw.more(); gw.next()) {
        const int row = uniform(rows[gw.grp]);
        const int mn = uniform(op.rmin[row]);
        const int S = uniform(op.rmax[row]) - mn + 1;
        const int a0 = uniform(op.Arp[row]), nA = uniform(op.Arp[row + 1]) - a0;
        const int tp = uniform(op.rtp[row]);
        const bool sparse = TL && use_sparse(S, tp);
        const int W = sparse ? (S + 63) >> 6 : S; // entries of the first level
        const StreamLayout L = sym_stream_layout(G, S, nA, tp);
        u64 *dm = (u64 *)lds;
        unsigned *doff = (unsigned *)(lds + L.doff);
        Stream<G> st;
        st.rec = (uint4 *)(lds + L.rec);
        st.bits = (u64 *)(lds + L.bits);
        st.wb = (unsigned short *)(lds + L.wb);
        st.red = red;
        const int words = (L.doff - L.bits) >> 3;
        const long long rd = op.dir_mask ? uniform64(op.rdir[row]) & ~RDIR_TWO : -1;
        auto tiles = [&](int e) { return tile_range(op, e, nA, op.Acol[a0 + e]); };
        // two-level rows walk their tiles twice: the lane's first entry is kept (with more lanes
        // that costs an R-MAT square of scale 18 0.5%)
        constexpr bool KEEP = TL && G <= 128;
        Segment mine = {0, 0, 0};
        if (KEEP && l < nA)
            mine = tiles(l);
        for (int t = l; t < W; t += G)
            dm[t] = 0;
        for (int q = l; q < words; q += G)
            st.bits[q] = 0;
        __syncthreads();
        auto walk_tiles = [&](auto body) {
            if constexpr (LONG)
                st.run(
                    nA, tile_range(op, l, nA, col_of(op, a0, l, nA)), [&](int e) { return col_of(op, a0, e, nA); },
                    [&](int e, int j) { return tile_range(op, e, nA, j); }, body);
            else
                st.run(nA, [&](int e) { return KEEP && e < G ? mine : tiles(e); }, body);
        };
        if (!sparse)
            walk_tiles([&](const Stream<G> &t, long long w0) {
                stream_or<G, OR_FLAT>(t, w0, op, dm, nullptr, nullptr, mn);
            });
        if constexpr (TL) {
            if (sparse)
                walk_tiles([&](const Stream<G> &t, long long w0) {
                    stream_or<G, OR_COARSE>(t, w0, op, dm, nullptr, nullptr, mn);
                });
        }
        const ChunkScan cs = scan_popcounts<G>(dm, W, (unsigned *)red);
        unsigned nnz = cs.tot;
        if (rd >= 0)
            for (int t = l; t < W; t += G)
                op.dir_mask[rd + t] = dm[t];
        __syncthreads();
        if (sparse)
            chunk_offsets<G>(dm, cs, [&](int t, unsigned p, u64) { doff[t] = p; });
        else if (rd >= 0)
            chunk_offsets<G>(dm, cs, [&](int t, unsigned p, u64) { dm[t] = p; });
        __syncthreads();
        if (rd >= 0)
            for (int t = l; t < W; t += G)
                op.dir_off[rd + t] = sparse ? doff[t] : (unsigned)dm[t];
        if constexpr (TL) {
            if (sparse) { // (uniform) the non-empty tiles' masks
                const int F = (int)cs.tot;
                u64 *fm = dm + W;
                for (int k = l; k < F; k += G)
                    fm[k] = 0;
                for (int q = l; q < words; q += G)
                    st.bits[q] = 0;
                __syncthreads();
                walk_tiles([&](const Stream<G> &t, long long w0) {
                    stream_or<G, OR_FINE>(t, w0, op, dm, doff, fm, mn);
                });
                const ChunkScan fs = scan_popcounts<G>(fm, F, (unsigned *)red);
                nnz = fs.tot;
                if (rd >= 0) {
                    for (int k = l; k < F; k += G)
                        op.dir_mask[rd + W + k] = fm[k];
                    __syncthreads();
                    chunk_offsets<G>(fm, fs, [&](int k, unsigned p, u64) { fm[k] = p; });
                    __syncthreads();
                    for (int k = l; k < F; k += G)
                        op.dir_off[rd + W + k] = (unsigned)fm[k];
                }
            }
        }
        if (l == 0)
            rnnz[row] = (int)nnz;
        __syncthreads();
    }
}

// Rows of the global bin whose flat directory does not fit LDS either (narrower ones run
// in k_symbolic_wide): the directory over the row's span in global memory, updated with
// L2 atomics -- in the kept directory (rdir) when the directories are kept, so the
// numeric phase reads masks and slot offsets from there, else in a per-workgroup
// workspace.  One 1024-lane workgroup per row.
__global__ __launch_bounds__(1024) void k_symbolic_global(const int *__restrict__ rows, const int *__restrict__ count_p,
                                                          Operands op, int *__restrict__ rnnz, int tshift, u64 *gws,
                                                          long long gws_stride)
{
    __shared__ unsigned red[16];
    const int l = threadIdx.x;
    const int nrows = *count_p;
    const int SG = 1 << tshift, sl = l & (SG - 1), sg = l >> tshift, NSG = 1024 >> tshift;
    for (int idx = blockIdx.x; idx < nrows; idx += gridDim.x) {
        const int row = rows[idx];
        const int mn = op.rmin[row];
        const int S = op.rmax[row] - mn + 1;
        const long long rd = op.dir_mask ? op.rdir[row] & ~RDIR_TWO : -1;
        u64 *dm = rd >= 0 ? op.dir_mask + rd : gws + (size_t)blockIdx.x * gws_stride;
        for (int t = l; t < S; t += 1024)
            dm[t] = 0;
        block_sync_global();
        const int a1 = op.Arp[row + 1];
        for (int e = op.Arp[row] + sg; e < a1; e += NSG) {
            const int j = op.Acol[e];
            const int t1 = op.tptr[j + 1];
            for (int t = op.tptr[j] + sl; t < t1; t += SG)
                atomicOr(&dm[op.tcol[t] - mn], op.tmask[t]);
        }
        block_sync_global();
        const ChunkScan cs = scan_popcounts<1024>(dm, S, red);
        if (rd >= 0)
            chunk_offsets<1024>(dm, cs, [&](int t, unsigned p, u64) { op.dir_off[rd + t] = p; });
        if (l == 0)
            rnnz[row] = (int)cs.tot;
        block_sync_global();
    }
}

// Rows of the global bin whose flat directory alone fits LDS (their staged A entries did
// not): the directory in LDS, B_j's tiles read from global memory per entry, as in
// k_symbolic_global, but ORed with ds_or_b64 instead of L2 atomics.  A kept directory
// goes out coalesced (masks, then the offsets written over them in LDS).  One 1024-lane
// workgroup per row; dynamic LDS: 8 bytes per tile of the widest span.
__global__ __launch_bounds__(1024) void k_symbolic_wide(const int *__restrict__ rows, const int *__restrict__ count_p,
                                                        Operands op, int *__restrict__ rnnz, int tshift)
{
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ unsigned red[16];
    u64 *dm = (u64 *)lds;
    const int l = threadIdx.x;
    const int nrows = *count_p;
    const int SG = 1 << tshift, sl = l & (SG - 1), sg = l >> tshift, NSG = 1024 >> tshift;
    for (int idx = blockIdx.x; idx < nrows; idx += gridDim.x) {
        const int row = uniform(rows[idx]);
        const int mn = uniform(op.rmin[row]);
        const int S = uniform(op.rmax[row]) - mn + 1;
        const long long rd = op.dir_mask ? uniform64(op.rdir[row]) & ~RDIR_TWO : -1;
        for (int t = l; t < S; t += 1024)
            dm[t] = 0;
        __syncthreads();
        const int a1 = op.Arp[row + 1];
        for (int e = op.Arp[row] + sg; e < a1; e += NSG) {
            const int j = op.Acol[e];
            or_walk<2 * UNROLL>(op, op.tptr[j], op.tptr[j + 1], SG, sl, dm, mn);
        }
        __syncthreads();
        const ChunkScan cs = scan_popcounts<1024>(dm, S, red);
        if (rd >= 0)
            for (int t = l; t < S; t += 1024)
                op.dir_mask[rd + t] = dm[t];
        __syncthreads();
        if (rd >= 0)
            chunk_offsets<1024>(dm, cs, [&](int t, unsigned p, u64) { dm[t] = p; });
        __syncthreads();
        if (rd >= 0)
            for (int t = l; t < S; t += 1024)
                op.dir_off[rd + t] = (unsigned)dm[t];
        if (l == 0)
            rnnz[row] = (int)cs.tot;
        __syncthreads();
    }
}

// ---- numeric -------------------------------------------------------------------------------

// C's entries of a row with a workgroup to itself (G = 64 to 1024 lanes): its B rows are
// walked as one element stream.  What bounds it: the L1's rate for loads (12 bytes per
// product; see the stream's loads), the LDS's for ds_add_f64 (24 cycles per 64 products),
// C's stores, and the chain of short phases of a row, which several workgroups per CU
// overlap (ablation on banded: staging and zeroing 130 us, adds 250, output 200 of 560).
// Against the walk it replaced (a sub-group of lanes per B row, 4- and 8-byte loads):
// banded 62,451 rows 594 -> 512 us of numeric time; R-MAT scale 16, compensated FP32, rows
// of 256 to 1024 lanes 1,950 -> 1,150 us; R-MAT scale 18, FP64, rows of 512 lanes 5.35 ->
// 3.31 ms.
// TL: some row of the launch has a two-level directory (the form costs registers, so
// launches without one run a kernel without it).  At 5 waves per SIMD (96 registers) ten
// banded rows of 128 lanes fit a CU as their LDS does.
template <int G, typename P, bool TL, bool LONG = false>
__global__ __launch_bounds__(G) __attribute__((amdgpu_waves_per_eu(TL ? 4 : 5))) void k_numeric_row(
    const int *__restrict__ rows, const int *__restrict__ count_p, Operands op, const long long *__restrict__ crp,
    int *__restrict__ Ccol, typename P::V *__restrict__ Cval, int *err, unsigned *queue)
{
    typedef typename P::V V;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ u64 red[16];
    __shared__ int grp_s[2];
    const int l = threadIdx.x;
    const V *__restrict__ Aval = (const V *)op.Aval;
    const int nrows = *count_p;
    for (GroupWalk gw(queue, nrows, grp_s, c_nxcd); gw.more(); gw.next()) {
        const int row = uniform(rows[gw.grp]);
        const int mn = uniform(op.rmin[row]);
        const int S = uniform(op.rmax[row]) - mn + 1;
        const long long cb = uniform64(crp[row]);
        const int n = (int)(uniform64(crp[row + 1]) - cb);
        const int a0 = uniform(op.Arp[row]), nA = uniform(op.Arp[row + 1]) - a0;
        const int tp = uniform(op.rtp[row]);
        const bool sparse = TL && use_sparse(S, tp);
        const int W = sparse ? (S + 63) >> 6 : S; // entries of the first level
        const StreamLayout L = stream_layout(G, S, n, nA, tp, uniform64(op.rprod[row]));
        double *vals = (double *)(lds + L.vals);
        u64 *dm = (u64 *)(lds + L.dm);
        unsigned *doff = (unsigned *)(lds + L.doff);
        unsigned *ft = (unsigned *)(lds + L.ft);
        Stream<G> st;
        st.rec = (uint4 *)(lds + L.rec);
        st.bits = (u64 *)(lds + L.bits);
        st.wb = (unsigned short *)(lds + L.wb);
        st.red = red;
        // fine level: the flat directory itself, or the compact entries after the coarse words
        u64 *fm = sparse ? dm + W : dm;
        unsigned *foff = sparse ? doff + W : doff;
        const bool dense = !sparse && use_dense(S, n);
        const int nv = dense ? 64 * S : n;
        const long long rd = op.dir_mask ? uniform64(kept_dir(op, row, sparse)) : -1;
        const int words = (L.doff - L.bits) >> 3;
        auto tiles = [&](int e) { return tile_range(op, e, nA, op.Acol[a0 + e]); };
        auto entry = [&](int e, int j) {
            if (e >= nA)
                return Segment{0, 0, 0};
            const typename Vec2<int>::type b = load2(op.Brp + j);
            const double a = (double)Aval[a0 + e];
            return Segment{b.x, b.y - b.x, (u64)__double_as_longlong(a)};
        };
        auto entries = [&](int e) { return entry(e, op.Acol[a0 + e]); };
        // two-level rows may walk their tiles twice and then their elements: the lane's first
        // entry is kept
        constexpr bool KEEP = TL && G <= 128;
        Segment my_tiles = {0, 0, 0}, mine = {0, 0, 0};
        if (KEEP && l < nA) {
            if (rd < 0)
                my_tiles = tiles(l);
            mine = entries(l);
        }
        for (int q = 2 * l; q < nv; q += 2 * G) // (the array is padded to 16 bytes)
            *(double2 *)(vals + q) = make_double2(0.0, 0.0);
        for (int q = l; q < words; q += G)
            st.bits[q] = 0;
        if (rd >= 0) { // directory kept by the symbolic phase: its first level
            for (int t = l; t < W; t += G) {
                dm[t] = op.dir_mask[rd + t];
                doff[t] = op.dir_off[rd + t];
            }
        } else {
            for (int t = l; t < W; t += G)
                dm[t] = 0;
        }
        __syncthreads();
        auto walk_tiles = [&](auto body) {
            if constexpr (LONG)
                st.run(
                    nA, tile_range(op, l, nA, col_of(op, a0, l, nA)), [&](int e) { return col_of(op, a0, e, nA); },
                    [&](int e, int j) { return tile_range(op, e, nA, j); }, body);
            else
                st.run(nA, [&](int e) { return KEEP && e < G ? my_tiles : tiles(e); }, body);
        };
        auto rezero = [&]() { // the stream's bits, for its next run
            __syncthreads();
            for (int q = l; q < words; q += G)
                st.bits[q] = 0;
        };
        // the first level: flat slot offsets or coarse compact indices, and its total
        unsigned tot = (unsigned)n;
        if (rd < 0) {
            if constexpr (TL) {
                if (sparse)
                    walk_tiles([&](const Stream<G> &t, long long w0) {
                        stream_or<G, OR_COARSE>(t, w0, op, dm, nullptr, nullptr, mn);
                    });
            }
            if (!sparse)
                walk_tiles([&](const Stream<G> &t, long long w0) {
                    stream_or<G, OR_FLAT>(t, w0, op, dm, nullptr, nullptr, mn);
                });
            rezero();
            const ChunkScan cs = scan_popcounts<G>(dm, W, (unsigned *)red);
            tot = cs.tot;
            chunk_offsets<G>(dm, cs, [&](int t, unsigned p, u64) { doff[t] = p; });
        } else if (sparse) {
            tot = W > 0 ? doff[W - 1] + (unsigned)__popcll(dm[W - 1]) : 0u;
        }
        unsigned nnz = tot;
        const int F = sparse ? (int)tot : S; // fine entries
        if (sparse) { // (uniform: one row per workgroup)
            __syncthreads();
            if (rd >= 0) {
                for (int k = l; k < F; k += G) {
                    fm[k] = op.dir_mask[rd + W + k];
                    foff[k] = op.dir_off[rd + W + k];
                }
                nnz = (unsigned)n;
            } else {
                for (int k = l; k < F; k += G)
                    fm[k] = 0;
            }
            // tile of every fine entry, from the coarse bitmap
            for (int w = l; w < W; w += G) {
                u64 m = dm[w];
                unsigned k = doff[w];
                while (m) {
                    ft[k++] = (unsigned)((w << 6) + __ffsll((unsigned long long)m) - 1);
                    m &= m - 1;
                }
            }
            __syncthreads();
            if (rd < 0) {
                walk_tiles([&](const Stream<G> &t, long long w0) {
                    stream_or<G, OR_FINE>(t, w0, op, dm, doff, fm, mn);
                });
                rezero();
                const ChunkScan fs = scan_popcounts<G>(fm, F, (unsigned *)red);
                nnz = fs.tot;
                chunk_offsets<G>(fm, fs, [&](int k, unsigned p, u64) { foff[k] = p; });
            }
        }
        const bool ok = (int)nnz == n;
        if (!ok && l == 0)
            raise_internal(err);
        __syncthreads();
        if (ok) { // uniform
            auto walk_rows = [&](auto body) {
                if constexpr (LONG)
                    st.run(
                        nA, entry(l, col_of(op, a0, l, nA)), [&](int e) { return col_of(op, a0, e, nA); }, entry, body);
                else
                    st.run(nA, [&](int e) { return KEEP && e < G ? mine : entries(e); }, body);
            };
            if (dense)
                walk_rows([&](const Stream<G> &t, long long w0) {
                    stream_add<G, SLOT_DENSE, P>(t, w0, op, nullptr, nullptr, fm, foff, vals, mn);
                });
            else if (!sparse)
                walk_rows([&](const Stream<G> &t, long long w0) {
                    stream_add<G, SLOT_FLAT, P>(t, w0, op, nullptr, nullptr, fm, foff, vals, mn);
                });
            if constexpr (TL) {
                if (sparse)
                    walk_rows([&](const Stream<G> &t, long long w0) {
                        stream_add<G, SLOT_TWO_LEVEL, P>(t, w0, op, dm, doff, fm, foff, vals, mn);
                    });
            }
            if (dense || (unsigned)n >= 16u * (unsigned)F) {
                // tiles holding 16 columns or more on average: a wave per tile, a lane per
                // column; OUT_U tiles' values are read before any is stored
                constexpr int NW = G / 64, OUT_U = 4;
                const int w = uniform(l >> 6), lane = l & 63;
                int *__restrict__ oc = Ccol + cb;
                V *__restrict__ ov = Cval + cb;
                for (int kb = w; kb < F; kb += 64 * NW) {
                    // lane i holds tile kb + i * NW
                    const int kt = kb + lane * NW;
                    u64 lm = 0;
                    unsigned lo = 0;
                    int lt = 0;
                    if (kt < F) {
                        lm = fm[kt];
                        lo = foff[kt];
                        lt = sparse ? (int)ft[kt] : kt;
                    }
                    const int left = (F - kb + NW - 1) / NW, cnt = left < 64 ? left : 64;
                    for (int i = 0; i < cnt; i += OUT_U) {
                        unsigned pos[OUT_U];
                        int col[OUT_U];
                        V val[OUT_U];
                        bool has[OUT_U];
#pragma unroll
                        for (int u = 0; u < OUT_U; ++u) {
                            const u64 m = readlane_u64(lm, i + u); // (0 past the last tile)
                            const int t = __builtin_amdgcn_readlane(lt, i + u);
                            has[u] = __builtin_amdgcn_inverse_ballot_w64(m);
                            pos[u] = (unsigned)__builtin_amdgcn_readlane((int)lo, i + u) + (unsigned)mbcnt(m);
                            col[u] = ((mn + t) << 6) + lane;
                            if (has[u])
                                val[u] = P::result(vals, dense ? (unsigned)((t << 6) + lane) : pos[u]);
                        }
#pragma unroll
                        for (int u = 0; u < OUT_U; ++u)
                            if (has[u]) {
                                oc[pos[u]] = col[u];
                                ov[pos[u]] = val[u];
                            }
                    }
                }
            } else { // a lane per tile, then the values in slot order
                for (int k = l; k < F; k += G) {
                    u64 m = fm[k];
                    unsigned pos = foff[k];
                    const int c0 = (mn + (sparse ? (int)ft[k] : k)) << 6;
                    while (m) {
                        Ccol[cb + pos] = c0 + __ffsll((unsigned long long)m) - 1;
                        ++pos;
                        m &= m - 1;
                    }
                }
                for (int q = l; q < n; q += G)
                    Cval[cb + q] = P::result(vals, q);
            }
        }
        __syncthreads();
    }
}

// Rows that do not fit LDS (wide rows): a dense accumulator over a window of WIN_COLS
// columns in LDS, slid over the row's column span.  One 1024-lane workgroup per row.  Every
// A entry e keeps, in a global workspace, a cursor into B_j (cur), the end of B_j (kend)
// and the column at the cursor (nxt).  For each window, the entries with nxt inside it are
// collected into an LDS list (ACT_CHUNK at a time), so an entry costs one coalesced load
// in a window it has nothing for; the listed entries' sub-groups walk B_j from the cursor
// while the columns stay in the window, adding each product into its slot (ds_add) and
// marking the column present (ds_or).  Every product is read once and sorted B rows need
// no search.  After a window its present columns are counted and written in column order
// after those of the previous windows.  (Reference: the spECK dense path of the wide-row
// bin, src/external/spECK/dense_acc.cu:3-267, whose early return leaves long rows
// unwritten.)
// Walk B_j from element k while the columns stay below chi, with a group of gw lanes of
// one wave (this lane is gl-th, the group starts at wave lane glo, gmask = gw one-bits):
// U elements per lane per step, all loads of a step issued before any is used.  B_j is
// sorted, so the in-window elements of a step are a prefix of its U * gw elements; add()
// takes each of them.  Returns the new cursor (the same in every lane of the group).
template <int U, typename V, typename F>
DEVI int walk_segment(const int *__restrict__ Bcol, const V *__restrict__ Bval, int k, int ke, int chi, int gw, int gl,
                      int glo, u64 gmask, F &&add)
{
    while (k < ke) {
        int c[U];
        V v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kk = k + gl + u * gw;
            c[u] = INT_MAX;
            v[u] = 0;
            if (kk < ke) {
                c[u] = Bcol[kk];
                v[u] = Bval[kk];
            }
        }
        int took = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = c[u] < chi;
            if (in)
                add(c[u], v[u]);
            took += __popcll((__ballot(in) >> glo) & gmask);
        }
        k += took;
        if (took < U * gw)
            break;
    }
    return k;
}

constexpr int WIN_COLS = 8192;
constexpr int WIN_WORDS = WIN_COLS / 64;
constexpr int ACT_CHUNK = 2048;
constexpr int WIN_LDS = WIN_COLS * 8 + WIN_WORDS * 8 + ACT_CHUNK * 4; // slots, presence bits, active list

// List the entries of [b0, min(b0 + ACT_CHUNK, nA)) whose next column is below chi: those
// with at least LONG_SEG elements of B_j left from the back of act (count *nlong), the
// others from the front (count *nact).  Every thread of the workgroup calls it.
DEVI void collect_active(const int *nxt, const int *cur, const int *kend, int b0, int nA, int chi, int *act, int *nact,
                         int *nlong)
{
    const int l = threadIdx.x, lane = l & 63;
    const int lim = b0 + ACT_CHUNK < nA ? b0 + ACT_CHUNK : nA;
    for (int e0 = b0; e0 < lim; e0 += 1024) {
        const int e = e0 + l;
        const bool live = e < lim && nxt[e] < chi;
        const bool lng = live && kend[e] - cur[e] >= LONG_SEG;
        const u64 ms = __ballot(live && !lng), ml = __ballot(lng);
        int s0 = 0, l0 = 0;
        if (lane == 0) {
            if (ms)
                s0 = atomicAdd(nact, __popcll(ms));
            if (ml)
                l0 = atomicAdd(nlong, __popcll(ml));
        }
        s0 = __shfl(s0, 0, 64);
        l0 = __shfl(l0, 0, 64);
        if (live && !lng)
            act[s0 + mbcnt(ms)] = e;
        if (lng)
            act[ACT_CHUNK - 1 - (l0 + mbcnt(ml))] = e;
    }
}

template <typename P>
__global__ __launch_bounds__(1024) void k_numeric_window(const int *__restrict__ rows, const int *__restrict__ count_p,
                                                         Operands op, const long long *__restrict__ crp,
                                                         int *__restrict__ Ccol, typename P::V *__restrict__ Cval,
                                                         int bshift, int *cur_ws, long long cur_stride, long long ft_stride,
                                                         int *err)
{
    typedef typename P::V V;
    const V *__restrict__ Aval = (const V *)op.Aval;
    const V *__restrict__ Bval = (const V *)op.Bval;
    extern __shared__ __align__(16) unsigned char lds[];
    double *acc = (double *)lds;
    u64 *bits = (u64 *)(lds + WIN_COLS * 8);
    int *act = (int *)(lds + WIN_COLS * 8 + WIN_WORDS * 8);
    __shared__ unsigned red[16];
    __shared__ unsigned woff[WIN_WORDS];
    __shared__ int nact_s, nlong_s;
    const int l = threadIdx.x, lane = l & 63, w = l >> 6;
    // per-workgroup workspace: cursors, ends of the B rows, columns at the cursors
    int *cur = cur_ws + (size_t)blockIdx.x * (3 * cur_stride + ft_stride);
    int *kend = cur + cur_stride;
    int *nxt = kend + cur_stride;
    const int SG = 1 << bshift, sl = l & (SG - 1), NSG = 1024 >> bshift;
    const int sg0 = lane & ~(SG - 1); // first lane of this lane's sub-group within the wave
    const u64 sgmask = SG >= 64 ? ~0ull : ((1ull << SG) - 1ull);
    const int nrows = *count_p;
    for (int idx = blockIdx.x; idx < nrows; idx += gridDim.x) {
        const int row = rows[idx];
        const int a0 = op.Arp[row], nA = op.Arp[row + 1] - a0;
        const long long cb = crp[row];
        const long long n = crp[row + 1] - cb;
        const int cbeg = op.rmin[row] << 6, cend = (op.rmax[row] + 1) << 6;
        for (int e = l; e < nA; e += 1024) {
            const int j = op.Acol[a0 + e];
            const int k0 = op.Brp[j], k1 = op.Brp[j + 1];
            cur[e] = k0;
            kend[e] = k1;
            nxt[e] = k0 < k1 ? op.Bcol[k0] : INT_MAX;
        }
        block_sync_global();
        long long written = 0;
        for (int c0 = cbeg; c0 < cend; c0 += WIN_COLS) {
            const int c1 = c0 + WIN_COLS;
            for (int q = l; q < WIN_COLS; q += 1024)
                acc[q] = 0.0;
            if (l < WIN_WORDS)
                bits[l] = 0;
            auto add_d = [&](int c, V v, double a) {
                const int q = c - c0;
                P::add(acc, (unsigned)q, a, v);
                atomicOr(&bits[q >> 6], 1ull << (q & 63));
            };
            for (int base = 0; base < nA; base += ACT_CHUNK) {
                if (l == 0) {
                    nact_s = 0;
                    nlong_s = 0;
                }
                __syncthreads();
                collect_active(nxt, cur, kend, base, nA, c1, act, &nact_s, &nlong_s);
                __syncthreads();
                const int nact = nact_s, nlong = nlong_s;
                for (int t = w; t < nlong; t += 16) {
                    const int e = act[ACT_CHUNK - 1 - t];
                    const int ke = kend[e];
                    const double a = (double)Aval[a0 + e];
                    const int k = walk_segment<4>(op.Bcol, Bval, cur[e], ke, c1, 64, lane, 0, ~0ull,
                                                  [&](int c, V v) { add_d(c, v, a); });
                    if (lane == 0) {
                        cur[e] = k;
                        nxt[e] = k < ke ? op.Bcol[k] : INT_MAX;
                    }
                }
                for (int t = l >> bshift; t < nact; t += NSG) {
                    const int e = act[t];
                    const int ke = kend[e];
                    const double a = (double)Aval[a0 + e];
                    const int k = walk_segment<2>(op.Bcol, Bval, cur[e], ke, c1, SG, sl, sg0, sgmask,
                                                  [&](int c, V v) { add_d(c, v, a); });
                    if (sl == 0) {
                        cur[e] = k;
                        nxt[e] = k < ke ? op.Bcol[k] : INT_MAX;
                    }
                }
                __syncthreads(); // act is rewritten by the next chunk
            }
            // column order: word offsets within the window, then one wave per word
            const unsigned cnt = l < WIN_WORDS ? (unsigned)__popcll(bits[l]) : 0u;
            unsigned tot;
            const unsigned pre = group_excl_scan<1024>(cnt, red, tot);
            if (l < WIN_WORDS)
                woff[l] = pre;
            __syncthreads();
            for (int q = w; q < WIN_WORDS; q += 16) {
                const u64 m = bits[q];
                const long long r = written + woff[q] + __popcll(m & below(lane));
                if (((m >> lane) & 1ull) && r < n) { // r >= n only if the counts disagree (flagged below)
                    Ccol[cb + r] = c0 + (q << 6) + lane;
                    Cval[cb + r] = P::result(acc, (unsigned)((q << 6) + lane));
                }
            }
            written += tot;
            __syncthreads();
        }
        if (l == 0 && written != n)
            raise_internal(err);
        block_sync_global(); // workspace of the next row
    }
}

// Wide rows whose tile directory was kept (flat, or two-level when the symbolic phase
// held the row in LDS): the HSMU compact accumulator, windowed over the row's OUTPUT
// positions.  A window is a run of directory entries [k0, k1) holding at most CW_VALS of
// C's entries and CW_TILES entries, so its slots and its part of the directory fit LDS;
// a column's slot is found in O(1) from the directory as in the LDS kernels (two-level
// rows read their coarse words, a few KiB per row, from global memory).  Cursors into
// the B rows and active lists as in the dense window kernel; a window spans the row's
// columns from its first to its last non-empty tile, so sparse stretches cost nothing and
// a row needs about max(nnz / CW_VALS, entries / CW_TILES) windows instead of span /
// WIN_COLS.  Values go out coalesced (they are C's entries in order), columns from the
// masks.
constexpr int CW_VALS = 4096;
constexpr int CW_TILES = 2048;
constexpr int CW_LDS = CW_VALS * 8 + CW_TILES * 16 + ACT_CHUNK * 4; // slots, window directory, active list

template <typename P>
__global__ __launch_bounds__(1024) void k_numeric_wcompact(const int *__restrict__ rows, const int *__restrict__ count_p,
                                                           Operands op, const long long *__restrict__ crp,
                                                           int *__restrict__ Ccol, typename P::V *__restrict__ Cval,
                                                           int bshift, int *ws, long long cur_stride, long long ft_stride,
                                                           int *err)
{
    typedef typename P::V V;
    const V *__restrict__ Aval = (const V *)op.Aval;
    const V *__restrict__ Bval = (const V *)op.Bval;
    extern __shared__ __align__(16) unsigned char lds[];
    double *vals = (double *)lds;
    u64 *wm = (u64 *)(lds + CW_VALS * 8);                        // window masks
    unsigned *wo = (unsigned *)(lds + CW_VALS * 8 + CW_TILES * 8); // slots relative to the window
    unsigned *wt = wo + CW_TILES;                                 // tiles relative to rmin
    int *act = (int *)(wt + CW_TILES);
    __shared__ int nact_s, nlong_s, k1_s;
    const int l = threadIdx.x, lane = l & 63, w = l >> 6;
    int *cur = ws + (size_t)blockIdx.x * (3 * cur_stride + ft_stride);
    int *kend = cur + cur_stride;
    int *nxt = kend + cur_stride;
    int *ft = nxt + cur_stride; // tile of every fine entry of a two-level row
    const int SG = 1 << bshift, sl = l & (SG - 1), NSG = 1024 >> bshift;
    const int sg0 = lane & ~(SG - 1);
    const u64 sgmask = SG >= 64 ? ~0ull : ((1ull << SG) - 1ull);
    const int nrows = *count_p;
    for (int idx = blockIdx.x; idx < nrows; idx += gridDim.x) {
        const int row = rows[idx];
        const int a0 = op.Arp[row], nA = op.Arp[row + 1] - a0;
        const long long cb = crp[row];
        const long long n = crp[row + 1] - cb;
        const int mn = op.rmin[row];
        const int S = op.rmax[row] - mn + 1;
        // the form the symbolic phase kept: two-level only if the row was in an LDS bin there
        const bool two = (op.rdir[row] & RDIR_TWO) != 0;
        const long long rd = op.rdir[row] & ~RDIR_TWO;
        const int W = two ? (S + 63) >> 6 : 0;
        const u64 *cmask = op.dir_mask + rd;      // coarse words (two-level)
        const unsigned *coff = op.dir_off + rd;
        const u64 *fm = op.dir_mask + rd + W;     // fine entries (flat: every tile of the span)
        const unsigned *foff = op.dir_off + rd + W;
        const int F = two ? (int)(coff[W - 1] + (unsigned)__popcll(cmask[W - 1])) : S;
        if (two) {
            for (int q = l; q < W; q += 1024) {
                u64 m = cmask[q];
                unsigned k = coff[q];
                while (m) {
                    ft[k++] = (q << 6) + __ffsll((unsigned long long)m) - 1;
                    m &= m - 1;
                }
            }
        }
        for (int e = l; e < nA; e += 1024) {
            const int j = op.Acol[a0 + e];
            const int k0 = op.Brp[j], k1 = op.Brp[j + 1];
            cur[e] = k0;
            kend[e] = k1;
            nxt[e] = k0 < k1 ? op.Bcol[k0] : INT_MAX;
        }
        block_sync_global();
        long long done = 0;
        for (int k0 = 0; k0 < F;) {
            // window end: at most CW_TILES entries and CW_VALS slots (one entry holds <= 64)
            if (l == 0) {
                const unsigned base = foff[k0];
                int lo = k0 + 1, hi = k0 + CW_TILES < F ? k0 + CW_TILES : F;
                while (lo < hi) { // largest k1 in [k0+1, hi] with slots(k0, k1) <= CW_VALS
                    const int mid = (lo + hi + 1) >> 1;
                    const long long end = mid == F ? n : (long long)foff[mid];
                    if (end - base <= CW_VALS)
                        lo = mid;
                    else
                        hi = mid - 1;
                }
                k1_s = lo;
            }
            __syncthreads();
            const int k1 = k1_s;
            const int nk = k1 - k0;
            const long long base = foff[k0];
            const int cnt = (int)((k1 == F ? n : (long long)foff[k1]) - base);
            for (int q = l; q < nk; q += 1024) {
                wm[q] = fm[k0 + q];
                wo[q] = (unsigned)(foff[k0 + q] - base);
                wt[q] = two ? (unsigned)ft[k0 + q] : (unsigned)(k0 + q);
            }
            for (int q = l; q < cnt; q += 1024)
                vals[q] = 0.0;
            __syncthreads();
            const int chi = (mn + (int)wt[nk - 1] + 1) << 6; // end of the window's last tile
            auto add_c = [&](int c, V v, double a) {
                const int tt = (c >> 6) - mn;
                const int ke2 = two ? (int)(coff[tt >> 6] + (unsigned)__popcll(cmask[tt >> 6] & below(tt & 63))) : tt;
                const int r = ke2 - k0;
                P::add(vals, wo[r] + (unsigned)__popcll(wm[r] & below(c & 63)), a, v);
            };
            for (int b0 = 0; b0 < nA; b0 += ACT_CHUNK) {
                if (l == 0) {
                    nact_s = 0;
                    nlong_s = 0;
                }
                __syncthreads();
                collect_active(nxt, cur, kend, b0, nA, chi, act, &nact_s, &nlong_s);
                __syncthreads();
                const int nact = nact_s, nlong = nlong_s;
                // long B rows: one wave each
                for (int t = w; t < nlong; t += 16) {
                    const int e = act[ACT_CHUNK - 1 - t];
                    const int ke = kend[e];
                    const double a = (double)Aval[a0 + e];
                    const int k = walk_segment<4>(op.Bcol, Bval, cur[e], ke, chi, 64, lane, 0, ~0ull,
                                                  [&](int c, V v) { add_c(c, v, a); });
                    if (lane == 0) {
                        cur[e] = k;
                        nxt[e] = k < ke ? op.Bcol[k] : INT_MAX;
                    }
                }
                // the others: sub-groups of SG lanes
                for (int t = l >> bshift; t < nact; t += NSG) {
                    const int e = act[t];
                    const int ke = kend[e];
                    const double a = (double)Aval[a0 + e];
                    const int k = walk_segment<2>(op.Bcol, Bval, cur[e], ke, chi, SG, sl, sg0, sgmask,
                                                  [&](int c, V v) { add_c(c, v, a); });
                    if (sl == 0) {
                        cur[e] = k;
                        nxt[e] = k < ke ? op.Bcol[k] : INT_MAX;
                    }
                }
                __syncthreads();
            }
            // C's entries of this window, in order
            for (int q = l; q < cnt; q += 1024)
                Cval[cb + base + q] = P::result(vals, (unsigned)q);
            for (int q = w; q < nk; q += 16) {
                const u64 m = wm[q];
                if ((m >> lane) & 1ull)
                    Ccol[cb + base + wo[q] + __popcll(m & below(lane))] = ((mn + (int)wt[q]) << 6) + lane;
            }
            done += cnt;
            k0 = k1;
            __syncthreads();
        }
        if (l == 0 && done != n)
            raise_internal(err);
        block_sync_global(); // workspace of the next row
    }
}

// ---- wide rows as windows -----------------------------------------------------------------

// The first element of [lo, hi) of a sorted row whose column is c or later.
DEVI int first_element(const int *__restrict__ col, int lo, int hi, int c)
{
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (col[mid] < c)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// The first element of every B row at each unit's start (and the row's end): index[j * (U + 1)
// + u] = first element of row j with a column of unit u or later.  A lane per (row, unit),
// binary search in the row (neighbouring lanes search one row).  In a replayed plan the row
// pointers are the inputs' current ones: without wide rows (as after a failed check of the
// plan) nothing is read, and what is read lies within B's nnz entries.
__global__ __launch_bounds__(256) void k_wide_index(const int *__restrict__ count_p, long long K, long long U, int nnz,
                                                    const int *__restrict__ rp, const int *__restrict__ col,
                                                    int *__restrict__ index)
{
    if (*count_p == 0)
        return;
    const long long n = K * (U + 1), stride = (long long)gridDim.x * 256;
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < n; q += stride) {
        const long long j = q / (U + 1), u = q - j * (U + 1);
        int lo = rp[j], hi = rp[j + 1];
        lo = lo < 0 ? 0 : lo < nnz ? lo : nnz;
        hi = hi < 0 ? 0 : hi < nnz ? hi : nnz;
        index[q] = u == 0 ? lo : u == U ? hi : first_element(col, lo, hi, (int)(u * WIDE_UNIT));
    }
}

constexpr int WI_BS = 1024; // lanes of a k_wide_items workgroup

// A wide row's directory in global memory, flat or two-level.
struct WideDir {
    const u64 *cm, *fm;
    const unsigned *co, *fo;
    int mn, S; // first tile, tiles spanned
    bool two;

    DEVI WideDir(const Operands &op, int first, int last, long long r)
    {
        mn = first;
        S = last - first + 1;
        two = (r & RDIR_TWO) != 0;
        const int W = two ? (S + 63) >> 6 : 0;
        const long long rd = r & ~RDIR_TWO;
        cm = op.dir_mask + rd;
        co = op.dir_off + rd;
        fm = cm + W;
        fo = co + W;
    }
    // entries of the (fine) level
    DEVI int entries() const
    {
        const int W = (S + 63) >> 6;
        return two ? (int)(uniform(co[W - 1]) + (unsigned)__popcll(uniform64(cm[W - 1]))) : S;
    }
    // entries of C_i, n of them in F = entries() tiles, before tile t (relative to mn, any
    // integer)
    DEVI unsigned before(int t, int F, unsigned n) const
    {
        if (t <= 0)
            return 0;
        if (t >= S)
            return n;
        int k = t;
        if (two) {
            k = (int)(co[t >> 6] + (unsigned)__popcll(cm[t >> 6] & below(t & 63)));
            if (k >= F)
                return n;
        }
        return fo[k];
    }
    // tile t's mask (0 outside the row's span) and the entries before it
    DEVI u64 tile(int t, unsigned &off) const
    {
        off = 0;
        if (t < 0 || t >= S)
            return 0;
        int k = t;
        if (two) {
            const u64 w = cm[t >> 6];
            if (!((w >> (t & 63)) & 1ull))
                return 0;
            k = (int)(co[t >> 6] + (unsigned)__popcll(w & below(t & 63)));
        }
        off = fo[k];
        return fm[k];
    }
};

// The windows of the wide rows, a wave per row: greedy runs of units.  FILL = false counts
// them per bucket (the heavy ones, then the compact and the dense form's by ranges of first
// units) and workgroup, FILL = true writes them, so that the list goes through C's columns
// in order and the workgroups that run together read the same part of B, which then stays in
// the L2s (R-MAT scale 18: 1/32 of B is 1.5 MB).  Bound by the chain of loads per row, so the grid fills the device.
template <bool FILL>
__global__ __launch_bounds__(WI_BS) void k_wide_items(const int *__restrict__ rows, const int *__restrict__ count_p,
                                                      Operands op, const long long *__restrict__ crp, long long U,
                                                      WideItem *__restrict__ items, long long cap,
                                                      unsigned *__restrict__ places, unsigned *__restrict__ hot,
                                                      long long hot_cap, long long hot_min, WideCount *ctr, int *err)
{
    __shared__ unsigned cnt[WIDE_LISTS]; // heavy windows, others, dense ones
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nrows = *count_p;
    unsigned *place = places + (size_t)threadIdx.x * gridDim.x + blockIdx.x; // bucket threadIdx.x's
    if (threadIdx.x < WIDE_LISTS)
        cnt[threadIdx.x] = FILL ? *place : 0u;
    __syncthreads();
    for (int i = blockIdx.x * (WI_BS / 64) + w; i < nrows; i += gridDim.x * (WI_BS / 64)) {
        const int row = uniform(rows[i]);
        const unsigned n = (unsigned)(uniform64(crp[row + 1]) - uniform64(crp[row]));
        const WideDir d(op, uniform(op.rmin[row]), uniform(op.rmax[row]), uniform64(op.rdir[row]));
        const int F = d.entries();
        const long long prod = uniform64(op.rprod[row]);
        const float work = (float)prod / (float)n; // products per entry of C_i
        const int nA = uniform(op.Arp[row + 1]) - uniform(op.Arp[row]);
        const int U0 = d.mn / WIDE_TILES, U1 = (d.mn + d.S - 1) / WIDE_TILES + 1; // units of the row
        int wu = 0, wv = 0; // lane i holds the i-th window found: its units [wu, wv) and
        unsigned wa = 0, we = 0; // the entries before its start and end
        int nw = 0;
        auto list = [&]() { // those found, a lane each
            if (lane < nw && we > wa) {
                const float p = work * (float)(we - wa);
                const bool dense = wv - wu == 1 && we - wa >= WIDE_DENSE && p < (float)WIDE_DENSE_WORK;
                const int b = (int)((long long)wu * WIDE_BUCKETS / U);
                const unsigned q =
                    atomicAdd(&cnt[p > (float)WIDE_HEAVY ? 0 : dense ? WIDE_LISTS - WIDE_BUCKETS + b : 1 + b], 1u);
                if (FILL) {
                    if (q < cap)
                        items[q] = WideItem{row, (unsigned)wu | ((unsigned)(wv - wu) << 24), wa, we - wa};
                    else // cannot happen: wide_row_items bounds them
                        raise_internal(err);
                    if (hot && q < cap && prod - (n - (we - wa)) > hot_min && (long long)nA * (we - wa) >= hot_min) {
                        const unsigned h = atomicAdd(&ctr->hot, 1u);
                        if (h < hot_cap) // (as above)
                            hot[h] = q;
                    }
                }
            }
            nw = 0;
        };
        int u = U0;      // first unit of the open window
        unsigned at = 0; // entries before it
        auto close = [&](int v, unsigned end) { // window [u, v)
            if (lane == nw) {
                wu = u;
                wv = v;
                wa = at;
                we = end;
            }
            u = v;
            at = end;
            if (++nw == 64)
                list();
        };
        unsigned prev = 0; // entries before unit vb - 1
        for (int vb = U0 + 1; vb <= U1; vb += 64) {
            const int v = vb + lane; // this lane's unit, and the entries before it
            const unsigned off = v < U1 ? d.before(v * WIDE_TILES - d.mn, F, n) : n;
            // the first unit that the open window cannot reach; a window has a unit at least
            // (which holds at most WIDE_UNIT entries), so u grows each time
            while (true) {
                const u64 m = __ballot(v > u + 1 && v <= U1 && (off - at > WIDE_UNIT || v - u > WIDE_UMAX));
                if (!m)
                    break;
                const int q = __ffsll((unsigned long long)m) - 1;
                close(vb + q - 1, q > 0 ? (unsigned)__builtin_amdgcn_readlane((int)off, q - 1) : prev);
            }
            prev = (unsigned)__builtin_amdgcn_readlane((int)off, 63);
        }
        close(U1, n);
        list();
    }
    __syncthreads();
    if (!FILL && threadIdx.x < WIDE_LISTS)
        *place = cnt[threadIdx.x];
}

// The place of each workgroup's first window in each bucket, from their numbers; the totals.
// One workgroup, in passes of 4,096 numbers.
__global__ __launch_bounds__(1024) void k_wide_order(unsigned *__restrict__ places, int groups, WideCount *ctr)
{
    __shared__ unsigned red[16], dense_s;
    const int n = WIDE_LISTS * groups, dense = (WIDE_LISTS - WIDE_BUCKETS) * groups;
    unsigned done = 0;
    for (int q0 = 0; q0 < n; q0 += 4096) {
        const int q = q0 + 4 * (int)threadIdx.x;
        unsigned k[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            k[i] = q + i < n ? places[q + i] : 0u;
        unsigned tot;
        unsigned at = done + group_excl_scan<1024>(k[0] + k[1] + k[2] + k[3], red, tot);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (q + i < n)
                places[q + i] = at;
            if (q + i == dense)
                dense_s = at;
            at += k[i];
        }
        done += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        ctr->dense = done - dense_s >= WIDE_DENSE_MIN ? dense_s : done;
        ctr->listed = done;
        ctr->taken[0] = ctr->taken[1] = 0;
        ctr->hot = ctr->sums = 0;
        ctr->parts = 0;
    }
}

// The elements of B's row j in units [u0, u1).
template <bool INDEX>
DEVI int2 window_elements(const Operands &op, const int *__restrict__ index, long long U, int u0, int u1, int j)
{
    if constexpr (INDEX) {
        const int *ix = index + (long long)j * (U + 1);
        return make_int2(ix[u0], ix[u1]);
    } else {
        const typename Vec2<int>::type r = load2(op.Brp + j);
        const int s0 = first_element(op.Bcol, r.x, r.y, u0 * WIDE_UNIT);
        return make_int2(s0, u1 < U ? first_element(op.Bcol, s0, r.y, u1 * WIDE_UNIT) : r.y);
    }
}

// The parts of hot windows that are this workgroup's: as k_numeric_windows' compact form, over a range
// of the row's entries.  Their sums meet by atomics in sum_val (k_wide_sums takes them to C); a
// window's first part writes its columns.
struct WideCut {
    const WidePart *parts;
    const WideCount *ctr;
    u64 part_cap;
    double *sum_val;
};
template <typename P, int BS, bool INDEX>
DEVI void window_parts(const WideCut &cut, const Operands &op, const int *__restrict__ index, long long U,
                       const long long *__restrict__ crp, int *__restrict__ Ccol, double *vals, Stream<BS> &st, u64 *wm,
                       unsigned short *wo)
{
    typedef typename P::V V;
    constexpr int NW = BS / 64, words = stream_window(BS) / 64;
    const int l = threadIdx.x, lane = l & 63, w = uniform((int)(threadIdx.x >> 6));
    const V *__restrict__ Aval = (const V *)op.Aval;
    const u64 n = cut.ctr->parts < cut.part_cap ? cut.ctr->parts : cut.part_cap;
    for (u64 i = blockIdx.x; i < n; i += gridDim.x) {
        const WidePart p = cut.parts[i];
        const int row = uniform(p.row), sum = uniform(p.sum), e0 = uniform(p.e0), cnt = (int)uniform(p.cnt);
        const unsigned units = uniform(p.units), base = uniform(p.base);
        const int u0 = (int)(units & 0xffffffu), u1 = u0 + (int)(units >> 24);
        const int a0 = uniform(op.Arp[row]) + e0, nA = uniform(p.e1) - e0;
        const WideDir d(op, uniform(op.rmin[row]), uniform(op.rmax[row]), uniform64(op.rdir[row]));
        const long long cb = uniform64(crp[row]) + base;
        const int T0 = u0 * WIDE_TILES, nt = (u1 - u0) * WIDE_TILES;
        for (int t = l; t < nt; t += BS) {
            unsigned off;
            wm[t] = d.tile(T0 + t - d.mn, off);
            wo[t] = (unsigned short)(off - base);
        }
        for (int q = 2 * l; q < cnt; q += 2 * BS) // (WIDE_UNIT is even)
            *(double2 *)(vals + q) = make_double2(0.0, 0.0);
        for (int q = l; q < words; q += BS)
            st.bits[q] = 0;
        __syncthreads();
        st.run(
            nA,
            [&](int e) {
                const int2 r = window_elements<INDEX>(op, index, U, u0, u1, op.Acol[a0 + e]);
                return Segment{r.x, r.y - r.x, (u64)__double_as_longlong((double)Aval[a0 + e])};
            },
            [&](const Stream<BS> &t, long long w0) {
                stream_add<BS, SLOT_FLAT, P>(t, w0, op, nullptr, nullptr, wm, wo, vals, T0);
            });
        __syncthreads();
        double *sv = cut.sum_val + (size_t)sum * WIDE_UNIT;
        for (int q = l; q < cnt; q += BS)
            unsafeAtomicAdd(&sv[q], vals[q]);
        if (e0 == 0)
            for (int t = w; t < nt; t += NW) {
                const u64 m = uniform64(wm[t]);
                if ((m >> lane) & 1ull)
                    Ccol[cb + wo[t] + (unsigned)mbcnt(m)] = ((T0 + t) << 6) + lane;
            }
        __syncthreads();
    }
}

// Wide rows as windows: the compact accumulator over one window's entries of C_i, its part
// of the row's directory (expanded to one mask and slot per tile of the window) and its
// elements of the B rows as one stream, their ranges read from the index or searched.  Workgroups
// take windows from the list until it is used up.  There are no atomics in C and no second round:
// a window's elements are known when it starts, and a window belongs to one workgroup.
// CUT: the parts of hot windows first, which then run beside the others.
// DENSE: a slot per column of the unit, with no masks in LDS: the element's column is its
// slot, and a tile goes out as one store of columns and one of values by a wave.
// No single unit bounds the compact form (Zipf panel: vector ALU 41%, LDS 32%, L1 47% of the
// time): a window's phases follow one another and 52 KB of LDS leave three workgroups per
// CU, so the next window's item, row and columns of A, and the next 256 entries' ranges, are
// loaded during the stream.  The dense form takes about a third fewer instructions and leaves
// room for four: Zipf panels of 2,000 rows 4.80 -> 4.25 ms, of 777 rows FP32 1.85 -> 1.55 ms
// (the calls; about 2.9 TB/s of C).
// The columns come from the window's masks: read from the directories in global memory by
// a kernel of its own they took 1.55 ms on the R-MAT square of scale 18.  Against items of up
// to 512 A entries that kept cursors into the B rows and posted chunks of them window by
// window (in rounds, with split rows meeting by atomics): scale 18 22.4 -> 8.6 ms, the Zipf
// panel 7.6 -> 3.9 ms.  With windows of up to 16 units (48 KB): compact form with 128 / 256 / 512
// lanes Zipf 6.3 / 4.8 / 5.0 ms, scale 18 20.8 / 17.4 / 17.5 ms; windows of 2,048 entries and twice
// the workgroups 6.1 and 18.4 ms.  Dense form with 512 lanes: Zipf 4.6 ms.
constexpr int WW_TILES = WIDE_TILES * WIDE_UMAX;
constexpr int WW_BS = 256; // lanes of a workgroup
constexpr int WW_PER_TILE = 16; // entries per tile from which a wave writes a tile's columns
template <int BS, bool DENSE> constexpr int ww_lds()
{
    constexpr int words = stream_window(BS) / 64;
    return WIDE_UNIT * 8 + BS * 16 + words * 10 + (DENSE ? 0 : WW_TILES * 10);
}
static_assert(3 * (ww_lds<WW_BS, false>() + LDS_STATIC_RESERVE) <= 160 * 1024, "three compact windows per CU");
static_assert(4 * (ww_lds<WW_BS, true>() + LDS_STATIC_RESERVE) <= 160 * 1024, "four dense windows per CU");

template <typename P, int BS, bool DENSE, bool INDEX, bool CUT = false>
__global__ __launch_bounds__(BS) void k_numeric_windows(const WideItem *__restrict__ items,
                                                        const WideCount *__restrict__ listed, unsigned *taken,
                                                        Operands op, const int *__restrict__ index, long long U,
                                                        const long long *__restrict__ crp, int *__restrict__ Ccol,
                                                        typename P::V *__restrict__ Cval, WideCut cut)
{
    typedef typename P::V V;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ u64 red[16];
    __shared__ unsigned next_s;
    constexpr int NW = BS / 64, words = stream_window(BS) / 64;
    double *vals = (double *)lds;
    Stream<BS> st;
    st.rec = (uint4 *)(vals + WIDE_UNIT);
    st.bits = (u64 *)(st.rec + BS);
    u64 *wm = st.bits + words;
    unsigned short *wo = (unsigned short *)(wm + (DENSE ? 0 : WW_TILES));
    st.wb = wo + (DENSE ? 0 : WW_TILES);
    st.red = red;
    int *stage = (int *)vals; // columns, once the values are out
    const int l = threadIdx.x, lane = l & 63, w = uniform((int)(threadIdx.x >> 6));
    const V *__restrict__ Aval = (const V *)op.Aval;
    if constexpr (CUT)
        window_parts<P, BS, INDEX>(cut, op, index, U, crp, Ccol, vals, st, wm, wo);
    const unsigned i0 = DENSE ? listed->dense : 0u, i1 = DENSE ? listed->listed : listed->dense;
    unsigned it = i0 + blockIdx.x;
    if (it >= i1)
        return;
    // a window's item, then its row's places, are loaded while the window before it is
    // worked on: raw loads here, made scalars (which waits for them) where they are used
    uint4 item = ((const uint4 *)items)[it];
    int row = uniform((int)item.x);
    int ra = op.Arp[row], rb = op.Arp[row + 1], rmn = op.rmin[row], rmx = op.rmax[row];
    long long rcb = crp[row], rrd = op.rdir[row];
    int j = l < rb - ra ? op.Acol[ra + l] : 0; // column of the lane's entry of A
    while (it < i1) {
        const unsigned units = uniform(item.y), base = uniform(item.z);
        const int cnt = (int)uniform(item.w);
        const int u0 = (int)(units & 0xffffffu), u1 = DENSE ? u0 + 1 : u0 + (int)(units >> 24);
        const int a0 = uniform(ra), nA = cnt ? uniform(rb) - a0 : 0; // (0: cut into parts)
        const WideDir d(op, uniform(rmn), uniform(rmx), uniform64(rrd));
        const long long cb = uniform64(rcb) + base;
        const int T0 = u0 * WIDE_TILES, nt = (u1 - u0) * WIDE_TILES;
        auto segment = [&](int e, int col) {
            if (e >= nA)
                return Segment{0, 0, 0};
            const int2 r = window_elements<INDEX>(op, index, U, u0, u1, col);
            return Segment{r.x, r.y - r.x, (u64)__double_as_longlong((double)Aval[a0 + e])};
        };
        const Segment first = segment(l, j);
        // dense: lane i of wave w holds tile w * TW + i
        constexpr int TW = WIDE_TILES / NW;
        u64 tm = 0;
        unsigned to = 0;
        if constexpr (DENSE) {
            tm = d.tile(T0 + w * TW + (lane < TW ? lane : TW - 1) - d.mn, to);
            tm = cnt ? tm : 0;
        } else {
            for (int t = l; t < nt; t += BS) {
                unsigned off;
                wm[t] = d.tile(T0 + t - d.mn, off);
                wo[t] = (unsigned short)(off - base);
            }
        }
        const int nv = DENSE ? WIDE_UNIT : cnt;
        for (int q = 2 * l; q < nv; q += 2 * BS) // (WIDE_UNIT is even)
            *(double2 *)(vals + q) = make_double2(0.0, 0.0);
        for (int q = l; q < words; q += BS)
            st.bits[q] = 0;
        if (l == 0)
            next_s = i0 + gridDim.x + atomicAdd(taken, 1u);
        __syncthreads();
        it = uniform(next_s);
        item = ((const uint4 *)items)[it < i1 ? it : i1 - 1];
        st.run(
            nA, first, [&](int e) { return e < nA ? op.Acol[a0 + e] : 0; }, segment,
            [&](const Stream<BS> &t, long long w0) {
                stream_add<BS, DENSE ? SLOT_DENSE : SLOT_FLAT, P>(t, w0, op, nullptr, nullptr, wm, wo, vals, T0);
            });
        row = uniform((int)item.x);
        ra = op.Arp[row];
        rb = op.Arp[row + 1];
        rmn = op.rmin[row];
        rmx = op.rmax[row];
        rcb = crp[row];
        rrd = op.rdir[row];
        int *cc = Ccol + cb;
        V *cv = Cval + cb;
        if constexpr (DENSE) { // a tile per step of a wave, a lane per column
#pragma unroll 4
            for (int i = 0; i < TW; ++i) {
                const u64 m = readlane_u64(tm, i);
                const unsigned q = (unsigned)__builtin_amdgcn_readlane((int)to, i) - base + (unsigned)mbcnt(m);
                const unsigned c = (unsigned)(w * TW + i) * 64 + lane;
                const V v = P::result(vals, c);
                if ((m >> lane) & 1ull) {
                    cc[q] = (T0 << 6) + (int)c;
                    cv[q] = v;
                }
            }
            j = l < rb - ra ? op.Acol[ra + l] : 0;
        } else {
            for (int q = l; q < cnt; q += BS)
                cv[q] = P::result(vals, (unsigned)q);
            j = l < rb - ra ? op.Acol[ra + l] : 0;
            // many entries per tile: a wave each, a lane per column; else a lane per tile and
            // LDS, for stores in order
            if (cnt >= WW_PER_TILE * nt) {
                for (int t = w; t < nt; t += NW) {
                    const u64 m = uniform64(wm[t]);
                    if ((m >> lane) & 1ull)
                        cc[wo[t] + (unsigned)mbcnt(m)] = ((T0 + t) << 6) + lane;
                }
            } else {
                __syncthreads();
                for (int t = l; t < nt; t += BS) {
                    u64 m = wm[t];
                    unsigned q = wo[t];
                    const int c = (T0 + t) << 6;
                    while (m) {
                        stage[q++] = c + __ffsll((unsigned long long)m) - 1;
                        m &= m - 1;
                    }
                }
                __syncthreads();
                for (int q = l; q < cnt; q += BS)
                    cc[q] = stage[q];
            }
        }
        __syncthreads();
    }
}

// Windows that may be hot, a wave each: the parts of those that are, which leave the list (no
// entries, no units).  An estimate that is off only makes the parts uneven; a window for whose
// parts or sums there is no room stays whole.
template <bool INDEX>
__global__ __launch_bounds__(256) void k_wide_cut(const unsigned *__restrict__ hot, unsigned hot_cap, long long hot_min,
                                                  WideItem *__restrict__ items, WideCount *ctr, Operands op,
                                                  const int *__restrict__ index, long long U,
                                                  const long long *__restrict__ crp, WidePart *__restrict__ parts,
                                                  u64 part_cap, WideSum *__restrict__ sums, double *__restrict__ sum_val,
                                                  unsigned sum_cap)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned n = ctr->hot < hot_cap ? ctr->hot : hot_cap;
    for (unsigned i = blockIdx.x * 4 + w; i < n; i += gridDim.x * 4) {
        const unsigned place = uniform(hot[i]);
        const WideItem it = items[place];
        const int row = uniform(it.row);
        const unsigned units = uniform(it.units), base = uniform(it.base), cnt = uniform(it.cnt);
        const int u0 = (int)(units & 0xffffffu), u1 = u0 + (int)(units >> 24);
        const int a0 = uniform(op.Arp[row]), nA = uniform(op.Arp[row + 1]) - a0;
        const int ns = nA < WIDE_SAMPLE ? nA : WIDE_SAMPLE;
        long long found = 0;
        for (int q = lane; q < ns; q += 64) {
            const int2 r = window_elements<INDEX>(op, index, U, u0, u1, op.Acol[a0 + (int)((long long)q * nA / ns)]);
            found += r.y - r.x;
        }
        const long long est = wave_sum(found) * nA / ns;
        if (est < hot_min)
            continue;
        const int by_na = nA / WIDE_PART_NA < WIDE_NA_PARTS ? nA / WIDE_PART_NA : WIDE_NA_PARTS;
        long long most = est / (hot_min / WIDE_PARTS);
        most = most > by_na ? most : by_na;
        most = most < nA ? most : nA;
        const int k = (int)(most < 4096 ? most : 4096);
        unsigned sum = 0;
        u64 at = 0;
        if (lane == 0) {
            sum = atomicAdd(&ctr->sums, 1u);
            if (sum < sum_cap)
                at = atomicAdd(&ctr->parts, (u64)k);
        }
        sum = uniform(sum);
        at = uniform64(at);
        if (sum >= sum_cap)
            continue;
        const bool fits = at + (u64)k <= part_cap;
        if (lane == 0)
            sums[sum] = WideSum{crp[row] + base, fits ? (long long)cnt : 0};
        if (!fits) { // (every place below ctr->parts is read)
            for (u64 q = at + lane; q < part_cap; q += 64)
                parts[q] = WidePart{row, (unsigned)u0, base, 0, 1, 1, (int)sum, 0};
            continue;
        }
        if (lane == 0)
            items[place] = WideItem{row, (unsigned)u0, base, 0};
        for (int q = lane; q < k; q += 64)
            parts[at + q] = WidePart{row, units, base, cnt, (int)((long long)nA * q / k), (int)((long long)nA * (q + 1) / k),
                                     (int)sum, 0};
        for (unsigned q = lane; q < cnt; q += 64)
            sum_val[(size_t)sum * WIDE_UNIT + q] = 0.0;
    }
}

template <typename P>
__global__ __launch_bounds__(256) void k_wide_sums(const WideSum *__restrict__ sums, const WideCount *__restrict__ ctr,
                                                   unsigned sum_cap, const double *__restrict__ sum_val,
                                                   typename P::V *__restrict__ Cval)
{
    const unsigned n = ctr->sums < sum_cap ? ctr->sums : sum_cap;
    for (unsigned i = blockIdx.x; i < n; i += gridDim.x)
        for (long long q = threadIdx.x; q < sums[i].cnt; q += 256)
            Cval[sums[i].at + q] = P::result(sum_val + (size_t)i * WIDE_UNIT, (unsigned)q);
}

// workgroups of a windows' kernel that a CU of lds_cu bytes holds
static int ww_per_cu(int lds, int lds_cu)
{
    const int n = lds_cu / (lds + LDS_STATIC_RESERVE);
    return n > 0 ? n : 1;
}

// ---- launchers -------------------------------------------------------------------------------

// Grid of an LDS row kernel: one workgroup per row group, or, with a work queue, as many
// workgroups as can be resident at once (occupancy for this LDS size x CUs).
template <typename Kern>
static int64_t row_grid(Kern kernel, int bs, size_t lds, int64_t groups, int num_cus, const unsigned *queue)
{
    int64_t blocks = groups;
    if (queue) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, bs, lds) != hipSuccess || per_cu < 1) {
            (void)hipGetLastError();
            per_cu = 1;
        }
        const int64_t resident = (int64_t)per_cu * (num_cus > 0 ? num_cus : 1);
        blocks = blocks < resident ? blocks : resident;
    }
    if (blocks > (1 << 20))
        blocks = 1 << 20;
    return blocks < 1 ? 1 : blocks;
}

// LDS of a row that shares a workgroup: the lanes of the workgroup's rows walk their slices
// in step, 8 bytes a lane, so slices an odd multiple of 8 G bytes apart keep them on
// different banks (padding that a small workgroup's LDS has room for).
template <int G> static int row_slice(int need)
{
    const int step = 8 * G, odd = ((need + step - 1) / step | 1) * step;
    return odd * (BLOCK / G) <= 32 * 1024 ? odd : (need + 15) & ~15;
}

// Waves per CU of a bin: a few times what is resident, so that a wave's start is paid for
// several groups of rows and the last ones to end are short.
constexpr int SMALL_WAVES = 128;
template <typename P, bool TOPS>
static hipError_t small_launch(const int *rows, long long stride, const BinStats *bins_dev, const int *count,
                               const BinStats &bins, const Operands &op, int *rnnz, const long long *crp, int *Ccol,
                               void *Cval, int *err, int num_cus, unsigned (*queue)[QUEUE_INTS],
                               unsigned long long *lds_bytes, hipStream_t s)
{
    SmallBins b = {};
    int64_t grid = 0;
    size_t lds = 0;
    for (int k = 0; k < BIN_SHARED; ++k) {
        if (count[k] <= 0)
            continue;
        const int rpb = BLOCK >> (k + 3), need = bins.max_need[k];
        b.rows[k] = rows + k * stride;
        b.count[k] = &bins_dev->count[k];
        b.queue[k] = queue ? queue[k] : nullptr;
        b.slice[k] = k == 0 ? row_slice<8>(need) : k == 1 ? row_slice<16>(need) : row_slice<32>(need);
        const size_t bytes = (size_t)b.slice[k] * rpb;
        lds = lds > bytes ? lds : bytes;
        const int64_t groups = ((int64_t)count[k] + rpb - 1) / rpb, most = (int64_t)SMALL_WAVES * num_cus;
        int64_t blocks = row_grid(k_small_rows<P, TOPS>, BLOCK, bytes, groups, num_cus, b.queue[k]);
        blocks = blocks < most ? blocks : most;
        // whole rounds over the XCDs, so that each bin's blocks start at the first
        b.blocks[k] = (int)((blocks + MAX_XCDS - 1) / MAX_XCDS * MAX_XCDS);
        grid += b.blocks[k];
        // a workgroup per group, as without the limit; a queue's workgroups are what runs
        *lds_bytes += (unsigned long long)(queue ? blocks : groups) * bytes;
    }
    if (grid == 0)
        return hipSuccess;
#define SMALL(B, G)                                                                                                    \
    if (b.blocks[B] == grid)                                                                                           \
        hipLaunchKernelGGL((k_small_bin<G, P, TOPS>), dim3((unsigned)grid), dim3(BLOCK), lds, s, b.rows[B], b.count[B],      \
                           b.slice[B], op, rnnz, crp, Ccol, (typename P::V *)Cval, err, b.queue[B]);                   \
    else
    SMALL(0, 8) SMALL(1, 16) SMALL(2, 32)
#undef SMALL
    hipLaunchKernelGGL((k_small_rows<P, TOPS>), dim3((unsigned)grid), dim3(BLOCK), lds, s, b, op, rnnz, crp, Ccol,
                       (typename P::V *)Cval, err);
    return hipGetLastError();
}

hipError_t launch_small(int form, const int *rows, long long stride, const BinStats *bins_dev, const int *count,
                        const BinStats &bins, const Operands &op, int *rnnz, const long long *crp, int *Ccol, void *Cval,
                        int *err, int num_cus, unsigned (*queue)[QUEUE_INTS], unsigned long long *lds_bytes, hipStream_t s)
{
    unsigned long long ignored = 0;
    if (!lds_bytes)
        lds_bytes = &ignored;
    bool tops = false; // a row may have a third level
    for (int k = 0; k < BIN_SHARED; ++k)
        tops |= count[k] > 0 && small_coarse(bins.max_span[k]) > SMALL_DIRECT;
    auto *f = form == SMALL_SYMBOLIC ? (tops ? small_launch<SmallNone, true> : small_launch<SmallNone, false>)
              : form == SMALL_F64    ? (tops ? small_launch<PrecF64, true> : small_launch<PrecF64, false>)
                                     : (tops ? small_launch<PrecF32C, true> : small_launch<PrecF32C, false>);
    return f(rows, stride, bins_dev, count, bins, op, rnnz, crp, Ccol, Cval, err, num_cus, queue, lds_bytes, s);
}

// Rows of 1,024 lanes that stage their entries in so many turns load the next turn's meanwhile.
constexpr int LONG_NA = 8 * 1024;

template <int G, bool TL, bool LONG = false>
static void symbolic_row(const int *rows, const int *count_dev, int count, int max_need, const Operands &op, int *rnnz,
                         int num_cus, unsigned *queue, hipStream_t s)
{
    const size_t lds = (size_t)((max_need + 15) & ~15);
    const int64_t blocks = row_grid(k_symbolic_row<G, TL, LONG>, G, lds, count, num_cus, queue);
    hipLaunchKernelGGL((k_symbolic_row<G, TL, LONG>), dim3((unsigned)blocks), dim3(G), lds, s, rows, count_dev, op, rnnz,
                       queue);
}

template <bool TL>
static void symbolic_rows(int bin, const int *rows, const int *count_dev, int count, int max_need, int max_na,
                          const Operands &op, int *rnnz, int num_cus, unsigned *queue, hipStream_t s)
{
    if (bin == NLDS - 1 && max_na >= LONG_NA) {
        symbolic_row<1024, TL, true>(rows, count_dev, count, max_need, op, rnnz, num_cus, queue, s);
        return;
    }
#define SYM(B, G)                                                                                                      \
    case B: symbolic_row<G, TL>(rows, count_dev, count, max_need, op, rnnz, num_cus, queue, s); break;
    switch (bin) {
        SYM(3, 64) SYM(4, 128) SYM(5, 256) SYM(6, 512) SYM(7, 1024)
    }
#undef SYM
}

hipError_t launch_symbolic(int bin, const int *rows, const int *count_dev, int count, int max_need, int max_na,
                           const Operands &op, int *rnnz, int tshift, int two_level, u64 *gws, long long gws_stride,
                           int num_cus, int gws_blocks, int lds_dyn, unsigned *queue, hipStream_t s)
{
    if (count <= 0)
        return hipSuccess;
    if (bin == BIN_GLOBAL) {
        const int blocks = count < gws_blocks ? count : gws_blocks;
        const size_t dir_lds = (size_t)gws_stride * sizeof(u64); // >= 8 bytes per tile of the widest span
        if (dir_lds <= (size_t)lds_dyn)
            hipLaunchKernelGGL(k_symbolic_wide, dim3(blocks), dim3(1024), dir_lds, s, rows, count_dev, op, rnnz,
                               tshift > 10 ? 10 : tshift);
        else
            hipLaunchKernelGGL(k_symbolic_global, dim3(blocks), dim3(1024), 0, s, rows, count_dev, op, rnnz,
                               tshift > 10 ? 10 : tshift, gws, gws_stride);
    } else if (bin >= BIN_SHARED && bin < NLDS) {
        if (two_level)
            symbolic_rows<true>(bin, rows, count_dev, count, max_need, max_na, op, rnnz, num_cus, queue, s);
        else
            symbolic_rows<false>(bin, rows, count_dev, count, max_need, max_na, op, rnnz, num_cus, queue, s);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int G, typename P, bool TL, bool LONG = false>
static void numeric_row(const int *rows, const int *count_dev, int count, int max_need, const Operands &op,
                        const long long *crp, int *Ccol, void *Cval, int *err, int num_cus, unsigned *queue,
                        unsigned long long *lds_bytes, hipStream_t s)
{
    const size_t lds = (size_t)((max_need + 15) & ~15);
    const int64_t blocks = row_grid(k_numeric_row<G, P, TL, LONG>, G, lds, count, num_cus, queue);
    *lds_bytes += (unsigned long long)blocks * lds;
    hipLaunchKernelGGL((k_numeric_row<G, P, TL, LONG>), dim3((unsigned)blocks), dim3(G), lds, s, rows, count_dev, op, crp,
                       Ccol, (typename P::V *)Cval, err, queue);
}

template <typename P, bool TL>
static void numeric_rows(int bin, const int *rows, const int *count_dev, int count, int max_need, int max_na,
                         const Operands &op,
                         const long long *crp, int *Ccol, void *Cval, int *err, int num_cus, unsigned *queue,
                         unsigned long long *lds_bytes, hipStream_t s)
{
    if (bin == NLDS - 1 && max_na >= LONG_NA) {
        numeric_row<1024, P, TL, true>(rows, count_dev, count, max_need, op, crp, Ccol, Cval, err, num_cus, queue,
                                       lds_bytes, s);
        return;
    }
#define NUM(B, G)                                                                                                      \
    case B:                                                                                                            \
        numeric_row<G, P, TL>(rows, count_dev, count, max_need, op, crp, Ccol, Cval, err, num_cus, queue, lds_bytes,   \
                              s);                                                                                      \
        break;
    switch (bin) {
        NUM(3, 64) NUM(4, 128) NUM(5, 256) NUM(6, 512) NUM(7, 1024)
    }
#undef NUM
}

template <typename P>
static hipError_t numeric_p(int bin, const int *rows, const int *count_dev, int count, int max_need, int max_na,
                            const Operands &op,
                            const long long *crp, int *Ccol, void *Cval, int bshift, int two_level,
                            const WideRows &wide, int *err, int num_cus, unsigned *queue,
                            unsigned long long *lds_bytes, hipStream_t s)
{
    if (bin == BIN_GLOBAL) {
        const int blocks = count < wide.blocks ? count : wide.blocks;
        if (op.dir_mask && wide.items) { // windows
            if (wide.index) {
                const long long gx = (wide.K * (wide.nunits + 1) + 255) / 256;
                hipLaunchKernelGGL(k_wide_index, dim3((unsigned)(gx < 65536 ? gx : 65536)), dim3(256), 0, s, count_dev,
                                   wide.K, wide.nunits, op.nnzB, op.Brp, op.Bcol, wide.index);
            }
            const unsigned gi = (unsigned)wide_item_blocks(count, num_cus);
            hipLaunchKernelGGL(k_wide_items<false>, dim3(gi), dim3(WI_BS), 0, s, rows, count_dev, op, crp, wide.nunits,
                               wide.items, wide.items_cap, wide.places, wide.hot, wide.hot_cap, wide.hot_min, wide.ctr, err);
            hipLaunchKernelGGL(k_wide_order, dim3(1), dim3(1024), 0, s, wide.places, (int)gi, wide.ctr);
            hipLaunchKernelGGL(k_wide_items<true>, dim3(gi), dim3(WI_BS), 0, s, rows, count_dev, op, crp, wide.nunits,
                               wide.items, wide.items_cap, wide.places, wide.hot, wide.hot_cap, wide.hot_min, wide.ctr, err);
            const unsigned gh = (unsigned)(8 * num_cus);
            const WideCut cut = {wide.parts, wide.ctr, (u64)wide.part_cap, wide.sum_val};
#define WINDOWS(DENSE, INDEX, CUT, TAKEN)                                                                              \
    hipLaunchKernelGGL((k_numeric_windows<P, WW_BS, DENSE, INDEX, CUT>),                                               \
                       dim3((unsigned)(num_cus * ww_per_cu(ww_lds<WW_BS, DENSE>(), wide.lds_cu))), dim3(WW_BS),        \
                       (ww_lds<WW_BS, DENSE>()), s, wide.items, wide.ctr, wide.ctr->taken + TAKEN, op, wide.index,     \
                       wide.nunits, crp, Ccol, (typename P::V *)Cval, cut)
#define FORM(INDEX)                                                                                                    \
    if (wide.hot)                                                                                                      \
        hipLaunchKernelGGL((k_wide_cut<INDEX>), dim3(gh), dim3(256), 0, s, wide.hot, (unsigned)wide.hot_cap,           \
                           wide.hot_min, wide.items, wide.ctr, op, wide.index, wide.nunits, crp, wide.parts,           \
                           (u64)wide.part_cap, wide.sums, wide.sum_val, (unsigned)wide.sum_cap);                       \
    WINDOWS(true, INDEX, false, 0);                                                                                    \
    if (wide.hot) {                                                                                                    \
        WINDOWS(false, INDEX, true, 1);                                                                                \
        hipLaunchKernelGGL(k_wide_sums<P>, dim3(gh), dim3(256), 0, s, wide.sums, wide.ctr, (unsigned)wide.sum_cap,     \
                           wide.sum_val, (typename P::V *)Cval);                                                       \
    } else {                                                                                                           \
        WINDOWS(false, INDEX, false, 1);                                                                               \
    }
            if (wide.index) {
                FORM(true)
            } else {
                FORM(false)
            }
#undef FORM
#undef WINDOWS
        } else if (op.dir_mask)
            hipLaunchKernelGGL(k_numeric_wcompact<P>, dim3(blocks), dim3(1024), CW_LDS, s, rows, count_dev, op, crp,
                               Ccol, (typename P::V *)Cval, bshift > 6 ? 6 : bshift, wide.ws, wide.cur_stride,
                               wide.ft_stride, err);
        else
            hipLaunchKernelGGL(k_numeric_window<P>, dim3(blocks), dim3(1024), WIN_LDS, s, rows, count_dev, op, crp, Ccol,
                               (typename P::V *)Cval, bshift > 6 ? 6 : bshift, wide.ws, wide.cur_stride, wide.ft_stride,
                               err);
    } else if (bin >= 3 && bin < NLDS) {
        if (two_level)
            numeric_rows<P, true>(bin, rows, count_dev, count, max_need, max_na, op, crp, Ccol, Cval, err, num_cus, queue,
                                  lds_bytes, s);
        else
            numeric_rows<P, false>(bin, rows, count_dev, count, max_need, max_na, op, crp, Ccol, Cval, err, num_cus, queue,
                                   lds_bytes, s);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_numeric(int bin, int fp32c, const int *rows, const int *count_dev, int count, int max_need, int max_na,
                          const Operands &op, const long long *crp, int *Ccol, void *Cval, int bshift, int two_level,
                          const WideRows &wide, int *err, int num_cus, unsigned *queue,
                          unsigned long long *lds_bytes, hipStream_t s)
{
    if (count <= 0)
        return hipSuccess;
    unsigned long long ignored = 0;
    if (!lds_bytes)
        lds_bytes = &ignored;
    if (fp32c)
        return numeric_p<PrecF32C>(bin, rows, count_dev, count, max_need, max_na, op, crp, Ccol, Cval, bshift, two_level, wide,
                                   err, num_cus, queue, lds_bytes, s);
    return numeric_p<PrecF64>(bin, rows, count_dev, count, max_need, max_na, op, crp, Ccol, Cval, bshift, two_level, wide, err,
                              num_cus, queue, lds_bytes, s);
}

int wide_item_blocks(int count, int num_cus)
{
    const int per = WI_BS / 64, most = 2 * num_cus; // 32 waves per CU
    return (count - 1) / per + 1 < most ? (count - 1) / per + 1 : most;
}

size_t wide_ws_ints(long long cur_stride, long long ft_stride, int blocks)
{
    return (size_t)blocks * (size_t)(3 * cur_stride + ft_stride);
}

hipError_t configure_kernels(int lds_max, int num_xcds)
{
    const int nx = num_xcds < 1 ? 1 : (num_xcds > MAX_XCDS ? MAX_XCDS : num_xcds);
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_nxcd), &nx, sizeof(int));
#define CFG(K)                                                                                                         \
    {                                                                                                                  \
        hipError_t r = hipFuncSetAttribute((const void *)(K), hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);    \
        if (r != hipSuccess)                                                                                           \
            e = r;                                                                                                     \
    }
#define CFGT(P, T)                                                                                                     \
    CFG((k_small_rows<P, T>)) CFG((k_small_bin<8, P, T>)) CFG((k_small_bin<16, P, T>)) CFG((k_small_bin<32, P, T>))
#define CFGL(P) CFGT(P, false) CFGT(P, true)
#define CFGS(TL)                                                                                                       \
    CFG((k_symbolic_row<64, TL>)) CFG((k_symbolic_row<128, TL>)) CFG((k_symbolic_row<256, TL>))                        \
    CFG((k_symbolic_row<512, TL>)) CFG((k_symbolic_row<1024, TL>)) CFG((k_symbolic_row<1024, TL, true>))
#define CFGR(P, TL)                                                                                                    \
    CFG((k_numeric_row<64, P, TL>)) CFG((k_numeric_row<128, P, TL>)) CFG((k_numeric_row<256, P, TL>))                  \
    CFG((k_numeric_row<512, P, TL>)) CFG((k_numeric_row<1024, P, TL>)) CFG((k_numeric_row<1024, P, TL, true>))
    CFGL(SmallNone) CFGL(PrecF64) CFGL(PrecF32C) CFGS(false) CFGS(true)
    CFGR(PrecF64, false) CFGR(PrecF32C, false) CFGR(PrecF64, true) CFGR(PrecF32C, true)
#undef CFGR
#undef CFGL
#undef CFGT
#undef CFGS
    CFG(k_symbolic_wide)
    CFG(k_numeric_window<PrecF64>) CFG(k_numeric_window<PrecF32C>)
    CFG(k_numeric_wcompact<PrecF64>) CFG(k_numeric_wcompact<PrecF32C>) 
#define CFGW(P)                                                                                                        \
    CFG((k_numeric_windows<P, WW_BS, false, false>)) CFG((k_numeric_windows<P, WW_BS, false, true>))                   \
    CFG((k_numeric_windows<P, WW_BS, true, false>)) CFG((k_numeric_windows<P, WW_BS, true, true>))                     \
    CFG((k_numeric_windows<P, WW_BS, false, false, true>)) CFG((k_numeric_windows<P, WW_BS, false, true, true>))
    CFGW(PrecF64) CFGW(PrecF32C)
#undef CFGW
#undef CFG
    return e;
}

} // namespace hsmu
