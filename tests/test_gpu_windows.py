"""Wide rows as windows of 4,096-column units: the edges of units and windows against the CPU
oracle (force_global sends every row there; lds_row_max sends those beyond it, whose
directories may be two-level)."""
import numpy as np
import pytest

import hsmu
import oracle

pytestmark = pytest.mark.gpu


def csr(rows, N, rng):
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate([np.sort(np.asarray(r, np.int64)) for r in rows]).astype(np.int32)
    return hsmu.HostMatrix(len(rows), N, rp, col, rng.uniform(-1, 1, len(col)).astype(np.float32).astype(np.float64))


def make(case):
    rng = np.random.default_rng(21)
    if case == "edges":  # first and last columns of units and of B
        N = 3 * 4096 + 1
        B = csr([[0, 4095, 4096, 8191], [8192, N - 1], [], [0], [N - 1], [4095, 4096], [1, 4097, 8193]], N, rng)
        A = csr([[0, 1, 6], [2], [3, 4], [5], list(range(7)), [0] * 300 + [4]], 7, rng)
    elif case == "full":  # units that are full: every window is one unit
        N = 4 * 4096 - 3
        B = csr([np.arange(0, N, 2), np.arange(1, N, 2), np.arange(N), [5, 5, 5]], N, rng)
        A = csr([[0, 1], [2], [0, 3], [0, 1, 2, 3] * 70], 4, rng)
    elif case == "span":  # few entries over many units: windows end at their span
        N = 4096 * 70
        B = csr([rng.choice(N, 40, replace=False) for _ in range(600)], N, rng)
        A = csr([rng.choice(600, n, replace=False) for n in (1, 255, 256, 257, 600)], 600, rng)
    else:  # single unit
        B = csr([rng.choice(100, n, replace=False) for n in rng.integers(0, 9, 50)], 100, rng)
        A = csr([rng.choice(50, n, replace=False) for n in (1, 50, 2, 30)], 50, rng)
    return A, B


@pytest.mark.parametrize("case", ["edges", "full", "span", "one"])
@pytest.mark.parametrize("opts", [dict(force_global=1), dict(lds_row_max=512), dict(force_global=1, rowptr64=1)])
@pytest.mark.parametrize("fp32", [False, True])
def test_windows(ctx, case, opts, fp32):
    A, B = make(case)
    print(f"[gpu-case] windows {case} {opts} fp32 {fp32}", flush=True)
    kw = dict(opts, precision=hsmu.HSMU_FP32_COMP) if fp32 else opts
    C, st = ctx.spgemm(A, B, **kw)
    ref = oracle.spgemm(A, B)
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
    assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)
    if "force_global" in opts:
        assert st["num_bin_rows"][8] == st["rows_nonempty"]


@pytest.mark.parametrize("N", [4093, 2 * 4096])  # a unit that ends within a tile; two per row
@pytest.mark.parametrize("fp32", [False, True])
def test_dense_windows(ctx, N, fp32):
    """Enough one-unit windows of at least 1,024 entries for the form with a slot per column,
    with some of fewer entries and of many products among them."""
    rng = np.random.default_rng(5)
    print(f"[gpu-case] dense windows N {N} fp32 {fp32}", flush=True)
    part = 1100 if N < 4096 else 5000
    B = csr([rng.choice(N, part, replace=False) for _ in range(20)] + [np.arange(N), [0], [N - 1], [], np.arange(0, N, 5)],
            N, rng)
    light = [[i % 20, 21 + i % 3] for i in range(8500)]
    A = csr(light + [[20], [24], [21, 22], [20] * 300, list(range(25)) * 30] + light[:300], 25, rng)
    C, _ = ctx.spgemm(A, B, force_global=1, precision=hsmu.HSMU_FP32_COMP if fp32 else hsmu.HSMU_FP64)
    ref = oracle.spgemm(A, B)
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
    assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)


@pytest.mark.parametrize("opts", [dict(), dict(rebuild_dirs=1), dict(wide_scratch_mb=1)])
def test_rows_of_64_kib(ctx, opts):
    """Rows around the LDS need from which they are cut into windows, with windows, without
    kept directories, and without room for the index (200 rows of B of 1,500 units)."""
    rng = np.random.default_rng(9)
    N = 4096 * 1500 if "wide_scratch_mb" in opts else 40000
    print(f"[gpu-case] rows of 64 KiB {opts}", flush=True)
    B = csr([rng.choice(40000, 100, replace=False) for _ in range(200)], N, rng)
    A = csr([rng.choice(200, n, replace=False) for n in (70, 78, 80, 82, 84, 90, 100, 150, 200)], 200, rng)
    C, st = ctx.spgemm(A, B, **opts)
    ref = oracle.spgemm(A, B)
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    assert np.all(np.abs(C.val - ref.val) <= 1e-12 * ref.absval)
    assert (st["num_bin_rows"][8] > 0) == (not opts)
