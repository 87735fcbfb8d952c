"""The one-pass conversion of B to tiles, the row analysis and the row pointers at the edges
of their blocks (2,048 entries; 1,024 rows; 256 blocks read back at a time; listed long
rows), against the CPU oracle: exact."""
import numpy as np
import pytest

import hsmu
import oracle

pytestmark = pytest.mark.gpu


def matrix(lens, N, rng, repeat=False):
    """Sorted rows of the given lengths: distinct columns, or a single repeated column."""
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    if repeat:
        col = np.repeat(rng.integers(0, N, len(lens)), lens)
    else:
        col = np.concatenate([np.sort(rng.choice(N, n, replace=False)) for n in lens] + [np.zeros(0)])
    return hsmu.HostMatrix(len(lens), N, rp, col.astype(np.int32), rng.integers(-3, 4, len(col)).astype(np.float64))


def lengths(case, rng):
    if isinstance(case, int):  # one entry per row but for a long first row: `case` entries in all
        return [min(case, 1500)] + [1] * max(0, case - 1500)
    return {"empty_rows": [0] * 5000 + [3] + [0] * 5000 + [2045, 0, 0, 7] + [0] * 2100,
            "chain": [17] * 40000,               # 333 blocks: more than one read back
            "long": [5000, 1, 4097, 0, 600, 4096] * 3}[case]


@pytest.mark.parametrize("case", [1, 2047, 2048, 2049, 4096, "empty_rows", "chain", "long"])
@pytest.mark.parametrize("repeat", [False, True])
def test_btiles_blocks(ctx, case, repeat):
    rng = np.random.default_rng(3)
    B = matrix(lengths(case, rng), 6000, rng, repeat)
    print(f"[gpu-case] btiles {case} repeat {repeat} nnz {B.nnz}", flush=True)
    for got, want in zip(ctx.btiles(B), oracle.btiles(B)):
        assert np.array_equal(got, want)


@pytest.mark.parametrize("M", [1, 127, 129, 1023, 1025, 2049, 70001])
def test_rows_and_row_pointers(ctx, M):
    rng = np.random.default_rng(M)
    lens = rng.integers(0, 4, M)
    lens[rng.integers(0, M, 3)] = [4500, 300, 130]  # listed rows: by a block, by a wave
    A = matrix(lens, 6000, rng)
    B = matrix(rng.integers(0, 3, 6000), 5000, rng)
    print(f"[gpu-case] rows {M}", flush=True)
    for wide in (0, 1):
        C, st = ctx.spgemm(A, B, rowptr64=wide)
        ref = oracle.spgemm(A, B)
        assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
        assert np.array_equal(C.val, ref.val)  # integers: exact
        assert st["products"] == oracle.products(A, B)
        assert sum(st["num_bin_rows"]) == sum(st["sym_bin_rows"])
