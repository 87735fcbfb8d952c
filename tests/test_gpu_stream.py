"""Rows with a workgroup to themselves walk their B rows as one stream of element pairs:
the edges of that stream against the CPU oracle (structure exact; FP64 within 1e-12 of
sum |a*b|, compensated FP32 within one FP32 rounding)."""
import numpy as np
import pytest

import hsmu
import oracle

pytestmark = pytest.mark.gpu


def csr(rows, N, rng):
    """Rows given as arrays of columns (repeats kept, sorted); values U(-1, 1) in FP32."""
    lens = [len(r) for r in rows]
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(np.asarray(r)) for r in rows]).astype(np.int32) if sum(lens) else np.zeros(0, np.int32)
    val = rng.uniform(-1, 1, len(col)).astype(np.float32).astype(np.float64)
    return hsmu.HostMatrix(len(rows), N, rp, col, val)


def make(case):
    rng = np.random.default_rng(7)
    if case == "one_entry":  # B holds a single entry: loads of two must not leave its arrays
        A = csr([[0] * 70, [0, 1], [1] * 65, []], 2, rng)
        return A, csr([[], [3]], 7, rng)
    if case == "odd_end":  # odd lengths, empty rows, an odd last row at the arrays' end
        B = csr([rng.choice(900, n, replace=False) for n in (0, 1, 2, 3, 64, 65, 127, 0, 129, 1)], 900, rng)
        A = csr([np.arange(10), [9] * 66, [0, 7], np.arange(1, 10, 2), np.repeat(np.arange(10), 13)], 10, rng)
        return A, B
    if case == "windows":  # more entries than lanes, more slots than a window, long rows of B
        B = csr([rng.integers(0, 4000, n) for n in [3] * 400 + [9001, 20000, 1] + [17] * 97], 4000, rng)
        A = csr([np.arange(500), rng.choice(500, 300, replace=False), [400, 401], [402] * 64], 500, rng)
        return A, B
    # sparse spans: two-level directories
    B = csr([rng.choice(1 << 20, n, replace=False) for n in rng.integers(0, 40, 300)], 1 << 20, rng)
    A = csr([rng.choice(300, n, replace=False) for n in (1, 2, 63, 64, 65, 200, 300)], 300, rng)
    return A, B


@pytest.mark.parametrize("case", ["one_entry", "odd_end", "windows", "sparse"])
@pytest.mark.parametrize("opts", [dict(products_per_lane=1), dict(products_per_lane=1, rebuild_dirs=1),
                                  dict(products_per_lane=64, lds_block_budget=64, persistent=1)])
@pytest.mark.parametrize("fp32", [False, True])
def test_stream(ctx, case, opts, fp32):
    A, B = make(case)
    print(f"[gpu-case] stream {case} {opts} fp32 {fp32}", flush=True)
    kw = dict(opts, precision=hsmu.HSMU_FP32_COMP) if fp32 else opts
    C, _ = ctx.spgemm(A, B, **kw)
    ref = oracle.spgemm(A, B)
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
    assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)
