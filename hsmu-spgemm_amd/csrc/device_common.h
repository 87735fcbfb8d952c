// device_common.h -- wave64 / workgroup helpers shared by the HIP kernel files.
#pragma once

#include <hip/hip_runtime.h>

#include "hsmu_internal.h"

namespace hsmu {

typedef unsigned long long u64;

#define DEVI __device__ __forceinline__

// ---- wave64 helpers ---------------------------------------------------------------

// number of set bits of m below this lane (v_mbcnt_lo/hi)
DEVI int mbcnt(u64 m)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

DEVI u64 below(int b) { return (1ull << b) - 1ull; }

// The first active lane's value, in a scalar register: for values that are the same in
// every lane (loaded from one address), so that no per-lane copy is kept.
DEVI int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
DEVI unsigned uniform(unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); }
DEVI long long uniform64(long long v)
{
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v & 0xffffffffLL));
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    return (long long)(((unsigned long long)hi << 32) | lo);
}
DEVI u64 uniform64(u64 v) { return (u64)uniform64((long long)v); }

// Lane k's value (k uniform), in scalar registers.
DEVI u64 readlane_u64(u64 v, int k)
{
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, k);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), k);
    return ((u64)hi << 32) | lo;
}

// One step of a scan over the wave: the value of the lane the DPP control names, or `none`
// where it names no lane (or the row mask leaves the row out).
template <int CTRL, int ROWS> DEVI unsigned dpp_step(unsigned none, unsigned v)
{
    return (unsigned)__builtin_amdgcn_update_dpp((int)none, (int)v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS> DEVI int dpp_step(int none, int v)
{
    return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS> DEVI u64 dpp_step(u64 none, u64 v)
{
    const unsigned lo = dpp_step<CTRL, ROWS>((unsigned)none, (unsigned)v);
    const unsigned hi = dpp_step<CTRL, ROWS>((unsigned)(none >> 32), (unsigned)(v >> 32));
    return ((u64)hi << 32) | lo;
}
template <int CTRL, int ROWS> DEVI long long dpp_step(long long none, long long v)
{
    return (long long)dpp_step<CTRL, ROWS>((u64)none, (u64)v);
}

// Inclusive scan over the 64 lanes (every lane must take part) with DPP moves: within rows
// of 16 lanes by 1, 2, 4, 8, then across rows.  No LDS round trip, unlike shuffles.
template <typename T, typename Op> DEVI T wave_incl_scan(T v, T none, Op op)
{
    v = op(v, dpp_step<0x111, 0xf>(none, v)); // row_shr:1
    v = op(v, dpp_step<0x112, 0xf>(none, v));
    v = op(v, dpp_step<0x114, 0xf>(none, v));
    v = op(v, dpp_step<0x118, 0xf>(none, v));
    v = op(v, dpp_step<0x142, 0xa>(none, v)); // row_bcast:15
    v = op(v, dpp_step<0x143, 0xc>(none, v)); // row_bcast:31
    return v;
}
template <typename T> DEVI T wave_incl_scan(T v)
{
    return wave_incl_scan(v, (T)0, [](T a, T b) { return a + b; });
}

DEVI unsigned wave_last(unsigned v) { return (unsigned)__builtin_amdgcn_readlane((int)v, 63); }
DEVI int wave_last(int v) { return __builtin_amdgcn_readlane(v, 63); }
DEVI u64 wave_last(u64 v) { return readlane_u64(v, 63); }
DEVI long long wave_last(long long v) { return (long long)readlane_u64((u64)v, 63); }

// Reductions over the 64 lanes (every lane must take part), the same in every lane.
template <typename T> DEVI T wave_sum(T v) { return wave_last(wave_incl_scan(v)); }
DEVI double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}
// of values that are not negative
DEVI int wave_max(int v)
{
    return wave_last(wave_incl_scan(v, 0, [](int a, int b) { return a > b ? a : b; }));
}

DEVI u64 wave_most(u64 v)
{
    return wave_last(wave_incl_scan(v, (u64)0, [](u64 a, u64 b) { return a > b ? a : b; }));
}

// Map the hardware block index so that each XCD (blocks are dealt round-robin over the
// nx XCDs of the device: 8 on an MI355X) works on a contiguous range of logical blocks:
// neighbouring rows, which share rows of B, then share one XCD's L2.
// (a division costs 20 vector instructions: nx is a power of two on full devices)
DEVI int xcd_block(int b, int n, int nx)
{
    int x, q, per, rem;
    if ((nx & (nx - 1)) == 0) {
        const int sh = __builtin_ctz(nx);
        x = b & (nx - 1);
        q = b >> sh;
        per = n >> sh;
        rem = n & (nx - 1);
    } else {
        x = b % nx;
        q = b / nx;
        per = n / nx;
        rem = n % nx;
    }
    return x * per + (x < rem ? x : rem) + q;
}

// Device work queue of the persistent row kernels: the n row groups of a launch are cut
// into nx contiguous ranges, one per XCD, each with a counter q[x * QUEUE_STRIDE] (zero at launch) that
// hands out chunks of `chunk` consecutive groups.  A workgroup takes the next chunk of its
// own XCD's range (xq starts at blockIdx.x % nx) and, once that range is used up, of the
// following ranges in turn, so the groups one XCD works on stay neighbours (shared rows
// of B in its L2) until the queues drain.  Thread 0 pulls; the chunk [s[0], s[1]) goes to
// every thread through LDS, s[0] = n when nothing is left.  The caller's loop body must
// end with a workgroup barrier before the next pull.
DEVI void pull_chunk(unsigned *q, int n, int chunk, int nx, int &xq, int *s)
{
    if (threadIdx.x == 0) {
        int got = n, end = n;
        for (int k = 0; k < nx; ++k) {
            const int x = (xq + k) % nx;
            const int lo = (int)((long long)n * x / nx), hi = (int)((long long)n * (x + 1) / nx);
            const unsigned nch = (unsigned)((hi - lo + chunk - 1) / chunk);
            if (__hip_atomic_load(&q[x * QUEUE_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= nch)
                continue;
            const unsigned v = atomicAdd(&q[x * QUEUE_STRIDE], 1u);
            if (v < nch) {
                got = lo + (int)v * chunk;
                end = got + chunk < hi ? got + chunk : hi;
                xq = x;
                break;
            }
        }
        s[0] = got;
        s[1] = end;
    }
    __syncthreads();
}

// The row groups a workgroup of a row kernel works on: with a queue, chunks pulled from
// it; without, groups xcd_block(block) + k * blocks (one group at a time).
// nx: XCDs of the device (1..MAX_XCDS).
struct GroupWalk {
    unsigned *q;
    int n, chunk, nx, xq, step, grp, end;
    int *s; // two ints of LDS

    // this workgroup is the block-th of `blocks` (all of the grid's, or a part of it)
    DEVI GroupWalk(unsigned *queue, int ngroups, int *lds2, int nxcd, int block = blockIdx.x, int blocks = gridDim.x)
        : q(queue), n(ngroups), chunk(1), nx(nxcd), xq(0), step(blocks), s(lds2)
    {
        if (q) {
            // chunks of about an eighth of a workgroup's share of its XCD's range
            const long long per = (long long)ngroups / ((long long)blocks * 8);
            chunk = per > 1 ? (int)per : 1;
            xq = block % nxcd;
            pull_chunk(q, n, chunk, nx, xq, s);
            grp = s[0];
            end = s[1];
        } else {
            grp = xcd_block(block, blocks, nx);
            end = grp + 1;
        }
    }
    DEVI bool more() const { return grp < n; }
    DEVI void next()
    {
        if (++grp < end)
            return;
        if (q) {
            pull_chunk(q, n, chunk, nx, xq, s);
            grp = s[0];
            end = s[1];
        } else {
            grp += step - 1;
            end = grp + 1;
        }
    }
};

// Reduction over a group of G <= 64 consecutive lanes, the same in every lane: with DPP
// moves up to 16 lanes (quad permutes, then the mirrors of half a row and of a row), which
// need no LDS; two shuffles at most beyond.
template <int G, typename T, typename Op> DEVI T group_reduce(T v, Op op)
{
    static_assert(G <= 64 && sizeof(T) <= 8, "a wave operation");
    if constexpr (G >= 2)
        v = op(v, dpp_step<0xB1, 0xf>(v, v)); // quad_perm:[1,0,3,2]
    if constexpr (G >= 4)
        v = op(v, dpp_step<0x4E, 0xf>(v, v)); // quad_perm:[2,3,0,1]
    if constexpr (G >= 8)
        v = op(v, dpp_step<0x141, 0xf>(v, v)); // row_half_mirror
    if constexpr (G >= 16)
        v = op(v, dpp_step<0x140, 0xf>(v, v)); // row_mirror
    if constexpr (G >= 32)
        v = op(v, __shfl_xor(v, 16, 64));
    if constexpr (G >= 64)
        v = op(v, __shfl_xor(v, 32, 64));
    return v;
}
template <int G, typename T> DEVI T group_sum(T v)
{
    return group_reduce<G>(v, [](T a, T b) { return a + b; });
}
template <int G, typename T> DEVI T group_min(T v)
{
    return group_reduce<G>(v, [](T a, T b) { return a < b ? a : b; });
}
template <int G, typename T> DEVI T group_max(T v)
{
    return group_reduce<G>(v, [](T a, T b) { return a > b ? a : b; });
}

// Exclusive scan over a group of G lanes; total = group sum.  G > 64 goes through LDS
// (every thread of the block must call it).
template <int G, typename T> DEVI T group_excl_scan(T v, T *red, T &total)
{
    constexpr int W = G < 64 ? G : 64;
    const int l = threadIdx.x & (W - 1);
    T x = v;
    if constexpr (G >= 64) {
        x = wave_incl_scan(v);
    } else { // (a shift within a row of 16 lanes also moves values between its groups)
        T y = dpp_step<0x111, 0xf>((T)0, x);
        x += l >= 1 ? y : (T)0;
        if constexpr (G >= 4) {
            y = dpp_step<0x112, 0xf>((T)0, x);
            x += l >= 2 ? y : (T)0;
        }
        if constexpr (G >= 8) {
            y = dpp_step<0x114, 0xf>((T)0, x);
            x += l >= 4 ? y : (T)0;
        }
        if constexpr (G >= 16) {
            y = dpp_step<0x118, 0xf>((T)0, x);
            x += l >= 8 ? y : (T)0;
        }
        if constexpr (G >= 32)
            x += dpp_step<0x142, 0xa>((T)0, x); // row_bcast:15
    }
    if constexpr (G == 64) {
        total = wave_last(x);
        return x - v;
    } else if constexpr (G < 64) {
        total = group_sum<G>(v);
        return x - v;
    } else {
        const int w = threadIdx.x >> 6;
        __syncthreads();
        if (l == 63)
            red[w] = x;
        __syncthreads();
        const int w0 = (threadIdx.x / G) * (G / 64);
        T before = 0, tot = 0;
#pragma unroll
        for (int k = 0; k < G / 64; ++k) {
            const T r = red[w0 + k];
            if (w0 + k < w)
                before += r;
            tot += r;
        }
        total = tot;
        return before + x - v;
    }
}

// Workgroup barrier that also orders global memory for the whole workgroup at device
// scope: prior stores are complete in L2 and this CU's L1 is invalidated afterwards,
// so plain loads see values other waves wrote with stores or L2 atomics.
DEVI void block_sync_global()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

} // namespace hsmu
