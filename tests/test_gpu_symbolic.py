"""Symbolic rows with a workgroup to themselves (a stream of tile pairs) and the form of the
directory they keep, against the CPU oracle (structure exact; values within 1e-12 of
sum |a*b|)."""
import numpy as np
import pytest

import hsmu
import oracle
from test_gpu_stream import make

pytestmark = pytest.mark.gpu


# lds_row_max 8 KiB: the two-level rows' flat directories are kept from global memory, and
# rows that fit only without the values take the wide path
@pytest.mark.parametrize("case", ["one_entry", "odd_end", "windows", "sparse"])
@pytest.mark.parametrize("opts", [dict(tiles_per_lane=1), dict(tiles_per_lane=1, rebuild_dirs=1),
                                  dict(tiles_per_lane=64, lds_block_budget=64, persistent=1),
                                  dict(lds_row_max=8192), dict(tiles_per_lane=1, lds_row_max=2048)])
def test_symbolic_rows(ctx, case, opts):
    A, B = make(case)
    print(f"[gpu-case] symbolic {case} {opts}", flush=True)
    C, _ = ctx.spgemm(A, B, **opts)
    ref = oracle.spgemm(A, B)
    assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
    assert np.all(np.abs(C.val - ref.val) <= 1e-12 * ref.absval)
