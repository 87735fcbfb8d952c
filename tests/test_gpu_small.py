"""Rows that share a wave (8, 16 or 32 lanes, elements in registers) at the limits of their
entries and pairs, against the CPU oracle (structure exact; FP64 within 1e-12 of sum |a*b|,
compensated FP32 within one FP32 rounding)."""
import numpy as np
import pytest

import hsmu
import oracle
from test_gpu_stream import csr

pytestmark = pytest.mark.gpu


def split(total, parts):
    """parts >= 1 lengths that add up to total, uneven."""
    cut = np.sort(np.random.default_rng(total * 97 + parts).choice(np.arange(1, total), parts - 1, replace=False)) if parts > 1 else []
    return np.diff(np.concatenate([[0], cut, [total]])).astype(int)


def make(N):
    rng = np.random.default_rng(N)
    rows_a, rows_b = [], []
    for nA in (1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33):
        for p in (nA, 63 - nA, 64 - nA, 65 - nA, 127 - nA, 128 - nA, 129 - nA, 255 - nA, 256 - nA, 257 - nA):
            if p < nA or p // nA > N:
                continue
            first = len(rows_b)
            for n in split(p, nA):  # (repeats allowed where the row is longer than B is wide)
                rows_b.append(rng.choice(N, n, replace=n > N))
            rows_a.append(np.arange(first, len(rows_b)))
    rows_b += [[], [N - 1]]  # the arrays' last element, alone in its row
    last = len(rows_b) - 1
    rows_a += [[], [last], [last - 1], [0, last - 1, last], [last] * 5, [last] * 40, [last - 1] * 20 + [0]]
    A = csr(rows_a, len(rows_b), rng)
    return A, csr(rows_b, N, rng)


@pytest.mark.parametrize("N", [1, 33, 700, 40000, 1 << 20])
@pytest.mark.parametrize("opts", [dict(products_per_lane=128, tiles_per_lane=128), dict(lds_block_budget=32768),
                                  dict(rebuild_dirs=1, persistent=1)])
@pytest.mark.parametrize("fp32", [False, True])
def test_small_rows(ctx, N, opts, fp32):
    A, B = make(N)
    print(f"[gpu-case] small rows N {N} {opts} fp32 {fp32}", flush=True)
    kw = dict(opts, precision=hsmu.HSMU_FP32_COMP) if fp32 else opts
    C, st = ctx.spgemm(A, B, **kw)
    ref = oracle.spgemm(A, B)
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
    assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)
    assert min(st["num_bin_rows"][:3]) > 0 or N == 1 << 20


@pytest.mark.parametrize("opts", [dict(), dict(rebuild_dirs=1), dict(force_global=1), dict(lds_block_budget=64)])
def test_rows_of_short_b(ctx, opts):
    """A B of short rows on average, whose tiles are made when a row of C wants them: rows of
    one lane group, a wave (over 64 entries) and a block (over 16,384) in B; rows of C that
    share waves, alone and beside rows that do not."""
    rng = np.random.default_rng(17)
    print(f"[gpu-case] short B {opts}", flush=True)
    N, K = 30000, 6000
    lens = rng.integers(0, 9, K)
    lens[[5, 255, 256, 4000]] = [65, 64, 16385, 300]
    lens[-1] = 7
    B = csr([rng.choice(N, n, replace=False) for n in lens], N, rng)
    assert len(B.col) <= 8 * K
    small = [rng.choice(np.arange(300, 3000), n, replace=False) for n in rng.integers(0, 8, 700)] + [[K - 1]]
    for rows in (small, small + [[5], [256, 5], np.arange(0, K, 7), [255, 4000]]):
        A = csr(rows, K, rng)
        C, st = ctx.spgemm(A, B, **opts)
        ref = oracle.spgemm(A, B)
        assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
        assert np.all(np.abs(C.val - ref.val) <= 1e-12 * ref.absval)
        tiles = sum(len(np.unique(np.asarray(B.col[B.rowptr[j]:B.rowptr[j + 1]]) >> 6)) for j in range(K))
        assert st["tiles_b"] == tiles
