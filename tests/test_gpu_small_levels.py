"""Rows that share a wave by their span: with no level above the words (a word or less per
product), with coarse words, and with a level above those (spans of more than 128 of them), at
the levels' edges; and rows of more than 32 entries of A, against the CPU oracle."""
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
    rng = np.random.default_rng(41)
    if case == "narrow":  # spans of 1..3 tiles, up to 240 products
        N, K = 191, 60
        B = csr([rng.integers(0, N if j % 2 else 64, rng.integers(0, 31)) for j in range(K)], N, rng)
        A = csr([rng.integers(0, K, rng.integers(0, 17)) for _ in range(3000)], K, rng)
    elif case == "words":  # spans of exactly a word per product and one more
        N, K = 64 * 130, 400
        B = csr([[64 * (j % 130), 64 * (j % 130) + j % 64] for j in range(K)], N, rng)
        A = csr([np.minimum(rng.integers(0, 100) + np.arange(k % 20 + 1) * rng.integers(1, 3), K - 1)
                 for k in range(2000)], K, rng)
    elif case in ("edges", "far edges"):  # columns around the borders of words, coarse and top words
        N, K = 1 << (22 if case == "edges" else 26), 300
        edge = np.concatenate([np.arange(-2, 2) + m for m in (32, 1024, 32768, 131072, 135168, 1 << 20, 1 << 25, N - 2)])
        edge = edge[(edge >= 0) & (edge < N)]
        B = csr([rng.choice(edge, rng.integers(1, 9), replace=False) for _ in range(K)], N, rng)
        A = csr([rng.choice(K, rng.integers(1, 33), replace=False) for _ in range(1500)], K, rng)
    elif case == "sparse":  # wide spans at random, 1..200 products
        N, K = 3000017, 2000
        B = csr([np.unique(rng.integers(0, N, rng.integers(0, 12))) for _ in range(K)], N, rng)
        A = csr([rng.choice(K, rng.integers(0, 28), replace=False) for _ in range(3000)], K, rng)
    elif case == "mixed":  # all the forms in one launch
        N, K = 1 << 20, 900
        B = csr([rng.integers(0, (64, 20000, N)[j % 3], 1 + j % 7) for j in range(K)], N, rng)
        A = csr([3 * rng.integers(0, K // 3, rng.integers(1, 30)) + (i % 3 if i % 4 else rng.integers(0, 3))
                 for i in range(3000)], K, rng)
    else:  # "long": 33 to 128 entries of A, one or no element each
        N, K = 70000, 5000
        B = csr([rng.integers(0, N, 1 if j % 5 else 0) for j in range(K)], N, rng)
        A = csr([rng.choice(K, n, replace=False) for n in (31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 140, 1) * 100], K, rng)
    return A, B


@pytest.mark.parametrize("case", ["narrow", "words", "edges", "far edges", "sparse", "mixed", "long"])
@pytest.mark.parametrize("opts", [dict(), dict(persistent=1), dict(timing=0, precision=hsmu.HSMU_FP32_COMP)])
def test_levels(ctx, case, opts):
    A, B = make(case)
    print(f"[gpu-case] small rows {case} {opts}", flush=True)
    C, st = ctx.spgemm(A, B, **opts)
    ref = oracle.spgemm(A, B)
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    fp32 = "precision" in opts
    bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
    assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)
    if case != "far edges":  # (top words of most of those rows exceed a wave's LDS)
        assert sum(st["num_bin_rows"][:3]) > st["rows_nonempty"] // 2
