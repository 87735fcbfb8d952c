"""Wide rows in the forms they take when the column index of B is not made (windows that search
B's rows), against the CPU oracle: unit edges as in test_gpu_windows.py, with rows of B added
that nothing names, so that the index would not pay; and what one hub row may cost."""
import numpy as np
import pytest

import hsmu
import oracle
from test_gpu_windows import csr, make

pytestmark = pytest.mark.gpu


def check(C, A, B, fp32=False):
    ref = oracle.spgemm(A, B)
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
    assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)


def more_rows(A, B, extra):
    """The same product with `extra` empty rows at the end of B."""
    rp = np.concatenate([B.rowptr, np.full(extra, B.rowptr[-1], np.int32)])
    return (hsmu.HostMatrix(A.M, A.N + extra, A.rowptr, A.col, A.val),
            hsmu.HostMatrix(B.M + extra, B.N, rp, B.col, B.val))


@pytest.mark.parametrize("case", ["edges", "full", "span", "one"])
@pytest.mark.parametrize("opts", [dict(force_global=1), dict(lds_row_max=512)])
@pytest.mark.parametrize("fp32", [False, True])
def test_windows_without_index(ctx, case, opts, fp32):
    A, B = more_rows(*make(case), 3000000)
    print(f"[gpu-case] windows without index {case} {opts} fp32 {fp32}", flush=True)
    C, st = ctx.spgemm(A, B, precision=hsmu.HSMU_FP32_COMP if fp32 else hsmu.HSMU_FP64, **opts)
    check(C, A, B, fp32)
    if "force_global" in opts:
        assert st["num_bin_rows"][8] == st["rows_nonempty"]


@pytest.mark.parametrize("fp32", [False, True])
def test_dense_windows_without_index(ctx, fp32):
    rng = np.random.default_rng(6)
    print(f"[gpu-case] dense windows without index fp32 {fp32}", flush=True)
    N = 2 * 4096 + 5
    B = csr([rng.choice(N, 2600, replace=False) for _ in range(20)] + [np.arange(N), [0], [N - 1], [4095, 4096], []],
            N, rng)
    A = csr([[i % 20, 20 + i % 5] if i % 50 else [i % 20, 21] for i in range(9000)] + [[20] * 200], 25, rng)
    A, B = more_rows(A, B, 20000000)
    C, st = ctx.spgemm(A, B, force_global=1, precision=hsmu.HSMU_FP32_COMP if fp32 else hsmu.HSMU_FP64)
    check(C, A, B, fp32)


def test_hub_row_takes_no_index():
    """A chain of 300,000 nodes, then with one node joined to 30,000 others: the hub adds its own
    entries of C and directory to the call's memory, not a place per row and 4,096 columns (90 MB)."""
    n, hub = 300000, 150000
    rng = np.random.default_rng(7)
    chain = [[j for j in (i - 1, i, i + 1) if 0 <= j < n] for i in range(n)]
    held = []
    for joined in (False, True):
        if joined:
            chain[hub] = np.unique(np.concatenate([chain[hub], rng.choice(n, 30000, replace=False)]))
        A = csr(chain, n, rng)
        print(f"[gpu-case] chain of {n}, hub {joined}", flush=True)
        ctx = hsmu.Context(0)
        try:
            C, st = ctx.spgemm(A, A)
            check(C, A, A)
            assert (st["num_bin_rows"][8] > 0) == joined
            held.append(hsmu.lib.hsmu_ctx_pool_bytes(ctx.handle))
        finally:
            ctx.close()
    assert held[1] - held[0] < 45e6


@pytest.mark.parametrize("fp32", [False, True])
def test_rows_that_fill_their_windows(ctx, fp32):
    """Rows of 130 KB of LDS at the span up to which they are cut into windows (a quarter full),
    and a tile wider, which stay in LDS."""
    rng = np.random.default_rng(13)
    N, n = 64 * 7600, 5000
    print(f"[gpu-case] rows at a quarter of their windows, fp32 {fp32}", flush=True)

    def row(tiles, first):  # n columns over exactly that many tiles
        inner = rng.choice(np.arange(first * 64 + 64, (first + tiles - 1) * 64), n - 2, replace=False)
        return np.concatenate([[first * 64 + 63], inner, [(first + tiles - 1) * 64]])

    B = csr([row(7500, 0), row(7501, 0), row(7500, 77), row(7501, 99)], N, rng)
    A = csr([[0], [1], [2], [3], [0], [3]], 4, rng)
    C, st = ctx.spgemm(A, B, precision=hsmu.HSMU_FP32_COMP if fp32 else hsmu.HSMU_FP64)
    check(C, A, B, fp32)
    assert st["num_bin_rows"][8] == 3 and st["rows_nonempty"] == 6
