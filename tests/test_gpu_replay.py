"""Replays of plans with wide rows on inputs whose structure changed: an error status and no
read outside the arrays, then the product again once the inputs are restored."""
import numpy as np
import pytest

import hsmu
import oracle

pytestmark = pytest.mark.gpu


def csr(rows, N, rng):
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate([np.sort(np.asarray(r, np.int64)) for r in rows]).astype(np.int32)
    return hsmu.HostMatrix(len(rows), N, rp, col, rng.uniform(-1, 1, len(col)))


def put(ctx, ptr, arr):
    arr = np.ascontiguousarray(arr, dtype=np.int32)
    hsmu._check(hsmu.lib.hsmu_copy_h2d(ctx.handle, ptr, arr.ctypes.data, arr.nbytes), "h2d")


def check(ctx, C, A, B):
    ref, got = oracle.spgemm(A, B), ctx.fetch(C)
    assert np.array_equal(np.asarray(got.rowptr, np.int64), ref.rowptr) and np.array_equal(got.col, ref.col)
    assert np.all(np.abs(got.val - ref.val) <= 1e-12 * ref.absval)


@pytest.mark.parametrize("count", [1, 2])  # a single product; a batch, whose B is stacked
def test_replay_wide_rows_changed_row_pointers(ctx, count):
    rng = np.random.default_rng(31)
    N = 4096 * 9
    pairs = []
    for _ in range(count):
        B = csr([rng.choice(N, 30, replace=False) for _ in range(400)], N, rng)
        A = csr([rng.choice(400, n, replace=False) for n in (3, 250, 257, 400)], 400, rng)
        pairs.append((A, B))
    dA, dB = [ctx.matrix(a) for a, _ in pairs], [ctx.matrix(b) for _, b in pairs]
    plan = ctx.plan(dA, dB, hsmu.default_opts(force_global=1))
    try:
        assert plan.execute()["num_bin_rows"][8] == 4 * count
        A, B = pairs[-1]
        far, back, less, order = (B.rowptr.copy() for _ in range(4))
        far[200] = 2 ** 31 - 1
        back[200] = -(2 ** 30)
        less[200] -= 7
        order[200], order[201] = order[201], order[200]
        for rp in (far, back, order, less):
            print(f"[gpu-case] replay of {count} with rowptr[200] = {rp[200]}", flush=True)
            put(ctx, dB[-1].rowptr, rp)
            try:
                plan.execute()
                assert rp is less  # in range and in order: only the rows' lengths changed
                check(ctx, plan.results[count - 1], A, hsmu.HostMatrix(B.M, B.N, rp, B.col, B.val))
            except hsmu.HsmuError as e:
                assert e.status in (hsmu.HSMU_ERR_PLAN, hsmu.HSMU_ERR_INDEX, hsmu.HSMU_ERR_UNSORTED)
            put(ctx, dB[-1].rowptr, B.rowptr)
            plan.execute()
            for C, (a, b) in zip(plan.results, pairs):
                check(ctx, C, a, b)
    finally:
        plan.destroy()
        for d in dA + dB:
            d.free()
