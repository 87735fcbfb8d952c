"""Wide rows with a window of many products, which is cut into ranges of the row's entries of A
whose sums meet in memory, against the CPU oracle: hot units, hot columns within a tile of a
window of many units, a unit that rows of B fill, beside rows that are not cut; with
and without the column index of B, and in a replayed plan."""
import numpy as np
import pytest

import hsmu
import oracle
from test_gpu_wide_forms import more_rows

pytestmark = pytest.mark.gpu


def make(case):
    rng = np.random.default_rng(61)
    if case == "unit":  # 2.4 M products in the second unit, some in every other
        K, per, N = 3000, 900, 4096 * 30
        col = rng.integers(0, N, (K, per))
        hot = rng.random((K, per)) < 0.9
        col[hot] = 4096 + rng.integers(0, 4096, int(hot.sum()))
        rows = [np.arange(K), np.arange(0, K, 3), np.arange(5), np.arange(K)]
    elif case == "tile":  # 60 columns of one tile in all rows of B, few others over 70 units
        K, N = 20000, 4096 * 70
        col = np.concatenate([np.tile(np.arange(64 * 101 + 2, 64 * 101 + 62), (K, 1)), rng.integers(0, N, (K, 3))], 1)
        rows = [np.arange(K), np.arange(1, K, 2), np.arange(17, 300)]
    else:  # "full": a unit that every row of B fills, by as many entries as it takes, one less, more
        K, N = 400, 4096 * 12 + 1
        col = np.concatenate([np.tile(np.arange(4096 * 3, 4096 * 4), (K, 1)), rng.integers(0, N, (K, 300))], 1)
        rows = [np.arange(128), np.arange(127), np.arange(129), np.arange(K), np.arange(0, K, 2)]
    col = np.sort(col, axis=1).astype(np.int32)
    K, per = col.shape
    val = lambda n: rng.uniform(-1, 1, n).astype(np.float32).astype(np.float64)
    B = hsmu.HostMatrix(K, N, (np.arange(K + 1) * per).astype(np.int32), col.ravel(), val(K * per))
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    A = hsmu.HostMatrix(len(rows), K, rp, np.concatenate(rows).astype(np.int32), val(rp[-1]))
    return A, B


def check(C, ref, fp32):
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
    assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)


@pytest.mark.parametrize("case", ["unit", "tile", "full"])
@pytest.mark.parametrize("indexed", [True, False])
@pytest.mark.parametrize("fp32", [False, True])
def test_hot_windows(ctx, case, indexed, fp32):
    A, B = make(case)
    if not indexed:
        A, B = more_rows(A, B, 2000000)
    ref = oracle.spgemm(A, B)
    o = hsmu.default_opts(force_global=1, precision=hsmu.HSMU_FP32_COMP if fp32 else hsmu.HSMU_FP64)
    dA, dB = ctx.matrix(A, fp32), ctx.matrix(B, fp32)
    print(f"[gpu-case] hot windows {case} indexed {indexed} fp32 {fp32}", flush=True)
    plan = ctx.plan([dA], [dB], o)
    try:
        check(ctx.fetch(plan.results[0]), ref, fp32)
        for _ in range(3):
            plan.execute()
            check(ctx.fetch(plan.results[0]), ref, fp32)
            C, _ = ctx.spgemm_device(dA, dB, o)
            check(ctx.fetch(C), ref, fp32)
            ctx.free_result(C)
    finally:
        plan.destroy()
        dA.free()
        dB.free()


def giant(case):
    rng = np.random.default_rng(71)
    if case == "narrow":  # a row that LDS holds, of most of the products; 14 tiles
        K, per, N, na = 200000, 4, 900, 200000
        col = rng.integers(0, N, (K, per))
    elif case == "spread":  # the same with a two-level directory
        K, per, N, na = 200000, 4, 1000000, 200000
        col = np.sort(rng.choice(N, 3000, replace=False))[rng.integers(0, 3000, (K, per))]
    else:  # "long": entries enough for the symbolic form without turns, products too few to be cut
        K, per, N, na = 60000, 3, 300000, 40000
        col = np.sort(rng.choice(N, 2000, replace=False))[rng.integers(0, 2000, (K, per))]
    col = np.sort(col, axis=1).astype(np.int32)
    val = lambda n: rng.uniform(-1, 1, n).astype(np.float32).astype(np.float64)
    B = hsmu.HostMatrix(K, N, (np.arange(K + 1) * per).astype(np.int32), col.ravel(), val(K * per))
    rows = [rng.choice(K, 5) for _ in range(700)]
    rows[300] = rng.choice(K, na, replace=False)
    rows = [np.sort(r) for r in rows]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    return hsmu.HostMatrix(len(rows), K, rp, np.concatenate(rows).astype(np.int32), val(rp[-1])), B


@pytest.mark.parametrize("case", ["narrow", "spread", "long"])
@pytest.mark.parametrize("fp32", [False, True])
def test_giant_rows(ctx, case, fp32):
    A, B = giant(case)
    ref = oracle.spgemm(A, B)
    o = hsmu.default_opts(precision=hsmu.HSMU_FP32_COMP if fp32 else hsmu.HSMU_FP64)
    dA, dB = ctx.matrix(A, fp32), ctx.matrix(B, fp32)
    print(f"[gpu-case] giant row {case} fp32 {fp32}", flush=True)
    plan = ctx.plan([dA], [dB], o)
    try:
        check(ctx.fetch(plan.results[0]), ref, fp32)
        for _ in range(3):
            plan.execute()
            check(ctx.fetch(plan.results[0]), ref, fp32)
        C, st = ctx.spgemm_device(dA, dB, o)
        check(ctx.fetch(C), ref, fp32)
        ctx.free_result(C)
        assert st["sym_bin_rows"][8] == 1 and st["num_bin_rows"][8] == (case != "long")
    finally:
        plan.destroy()
        dA.free()
        dB.free()
