// The host orchestrator (api.cpp) with the device replaced: memory is the host's, blocks beyond
// a limit cannot be had, and launches only write the counters of one product with wide rows.
// Checks which form those rows take as memory runs out, in a plan's two passes.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../hsmu-spgemm_amd/csrc/hsmu_internal.h"
#include "../../include/hsmu.h"

using namespace hsmu;

static size_t g_limit;      // bytes of a block that can be had
static long long g_blocks;  // blocks held
static DevStats g_stats[2]; // the counters at the two checkpoints
static std::vector<WideRows> g_wide;

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    if (n > g_limit)
        return hipErrorOutOfMemory;
    *p = malloc(n);
    ++g_blocks;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    free(p);
    --g_blocks;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 8;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int)
{
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 160 * 1024;
    p->totalGlobalMem = 288ull << 30;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    *g = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t)
{
    *t = 0;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = nullptr;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
}

namespace hsmu {
#define LAUNCH(name, ...)                                                                                              \
    hipError_t name(__VA_ARGS__) { return hipSuccess; }
typedef const int *ci;
typedef unsigned long long u64;
LAUNCH(launch_fill_zero, void *, size_t, hipStream_t)
LAUNCH(launch_copy, const void *, void *, size_t, int, hipStream_t)
LAUNCH(launch_brows, int64_t, int64_t, int64_t, ci, ci, BRow *, DevStats *, int, hipStream_t)
LAUNCH(launch_pad_b, ci, const void *, int, int, int *, void *, hipStream_t)
LAUNCH(launch_small, int, ci, long long, const BinStats *, ci, const BinStats &, const Operands &, int *, const long long *, int *,
       void *, int *, int, unsigned (*)[QUEUE_INTS], u64 *, hipStream_t)
LAUNCH(launch_btiles, int64_t, int64_t, int64_t, ci, ci, int *, int *, u64 *, BRow *, u64 *, unsigned *, DevStats *,
       hipStream_t)
LAUNCH(launch_symbolic, int, ci, ci, int, int, int, const Operands &, int *, int, int, u64 *, long long, int, int, int,
       unsigned *, hipStream_t)
LAUNCH(launch_row_sums, int64_t, const void *, int, const void *, int, double *, double *, hipStream_t)
LAUNCH(launch_plan_bases, const long long *, const long long *, int64_t, DevStats *, hipStream_t)
LAUNCH(launch_plan_check, DevStats *, const DevStats *, int, hipStream_t)
LAUNCH(launch_batch_split, int64_t, BatchOffsets, const long long *, void *, int, long long *, int64_t, hipStream_t)
LAUNCH(launch_batch_rowptr, int, int64_t, const BatchInst *, BatchOffsets, int64_t, int64_t, int *, DevStats *,
       hipStream_t)
LAUNCH(launch_batch_entries, int, int64_t, const BatchInst *, BatchOffsets, int64_t, int, int *, int *, void *,
       DevStats *, hipStream_t)
LAUNCH(launch_rowptr_narrow, const long long *, int64_t, int *, hipStream_t)
LAUNCH(launch_rowptr_rebase, ci, int64_t, int *, hipStream_t)
LAUNCH(configure_kernels, int, int)
LAUNCH(scratch_setup, int, void **)
int64_t btiles_blocks(int64_t) { return 1; }
int64_t rowptr_blocks(int64_t) { return 1; }
int wide_item_blocks(int, int) { return 1; }
size_t wide_ws_ints(long long cur, long long ft, int blocks) { return (size_t)blocks * (size_t)(3 * cur + ft); }
std::mutex &scratch_lock(int)
{
    static std::mutex m;
    return m;
}
static hipError_t counters(HostStats *host, unsigned seq, int k)
{
    if (host) {
        host->st = g_stats[k];
        host->seq = seq;
    }
    return hipSuccess;
}
hipError_t launch_row_info(int64_t, int64_t, int64_t, ci, ci, const BRow *, ci, long long *, int *, int *, int *, int *,
                           BinParams, int *, long long *, DevStats *, BinSum *, unsigned *, HostStats *host,
                           unsigned seq, int, hipStream_t)
{
    return counters(host, seq, 0);
}
hipError_t launch_rowptr_bin(int64_t, ci, const long long *, ci, ci, ci, ci, long long *, int *, BinParams, int *, u64 *,
                             unsigned *, DevStats *, BinSum *, unsigned *, HostStats *host, unsigned seq, hipStream_t)
{
    return counters(host, seq, 1);
}
hipError_t launch_numeric(int bin, int, ci, ci, int, int, int, const Operands &, const long long *, int *, void *, int, int,
                          const WideRows &w, int *, int, unsigned *, u64 *, hipStream_t)
{
    if (bin == BIN_GLOBAL)
        g_wide.push_back(w);
    return hipSuccess;
}
} // namespace hsmu

int main()
{
    hsmu_ctx *ctx = nullptr;
    g_limit = SIZE_MAX;
    if (hsmu_ctx_create(0, &ctx) != HSMU_OK)
        return 1;
    // 4 wide rows; a B of 2^20 rows and 15 units: an index of 64 MiB, other blocks of 16 at most
    int zero[2] = {0, 0};
    double one[2] = {1, 1};
    hsmu_csr A = {4, 1 << 20, 2, zero, zero, one, 0, 0}, B = {1 << 20, 4096 * 15, 2, zero, zero, one, 0, 0};
    struct {
        const char *what;
        size_t limit;
        unsigned long long items;
        int na, form; // 0: index, 1: search, 2: a workgroup per row, 3: no memory
    } cases[] = {{"all", SIZE_MAX, 64, 100, 0},
                 {"no index", 32 << 20, 64, 100, 1},
                 {"no index, no lists", 32 << 20, 4 << 20, 100, 2},
                 {"nothing", 32 << 20, 4 << 20, 1 << 20, 3},
                 {"all again", SIZE_MAX, 64, 100, 0}};
    for (auto &t : cases) {
        memset(g_stats, 0, sizeof(g_stats));
        g_stats[0].dir_total = 4096;
        g_stats[0].num_wide_work = g_stats[1].num.work[BIN_GLOBAL] = 1ull << 30;
        g_stats[0].sym.count[NLDS - 1] = g_stats[1].num.count[BIN_GLOBAL] = 4;
        g_stats[1].num.nnz_a[BIN_GLOBAL] = 1 << 24;
        g_stats[1].num.max_na[BIN_GLOBAL] = t.na;
        g_stats[1].num.max_span[BIN_GLOBAL] = 960;
        g_stats[1].wide_items = t.items;
        g_stats[1].hot_items = 16 << 20; // a list of 64 MiB
        g_stats[1].hot_most = 1ull << 30;
        g_stats[1].nnz_c = 1000;
        hsmu_ctx_trim(ctx);
        g_limit = t.limit;
        g_wide.clear();
        hsmu_opts o;
        hsmu_opts_default(&o);
        hsmu_plan *plan = nullptr;
        hsmu_csr C;
        const int rc = hsmu_plan_create(ctx, 1, &A, &B, &C, &o, &plan);
        bool ok = (rc == HSMU_ERR_NOMEM) == (t.form == 3) && (rc == HSMU_OK) == (t.form < 3);
        ok = ok && g_wide.size() == (t.form < 3 ? 2u : 0u);
        for (const WideRows &w : g_wide) // recording, capture: the same form in the same blocks
            ok = ok && (w.items != nullptr) == (t.form < 2) && (w.index != nullptr) == (t.form == 0) &&
                 (w.hot != nullptr) == (t.form == 0) && w.hot == g_wide[0].hot && w.sum_val == g_wide[0].sum_val &&
                 (t.form != 2 || w.ws) && w.items == g_wide[0].items && w.index == g_wide[0].index &&
                 w.ws == g_wide[0].ws && w.ctr == g_wide[0].ctr;
        hsmu_plan_destroy(plan);
        printf("%s: status %d, %s\n", t.what, rc, ok ? "ok" : "WRONG");
        if (!ok)
            return 1;
    }
    hsmu_ctx_destroy(ctx);
    if (g_blocks != 0)
        return 1;
    printf("WIDE_MEMORY_OK\n");
    return 0;
}
