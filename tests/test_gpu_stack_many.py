"""Stacking of many small instances, more than 16 to a chunk of 4,096 places and, with empty
ones among them, more than there are places, against the CPU oracle."""
import numpy as np
import pytest

import hsmu
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("same", [True, False])
@pytest.mark.parametrize("opts", [dict(), dict(rowptr64=1, precision=hsmu.HSMU_FP32_COMP)])
def test_many_instances(ctx, same, opts):
    rng = np.random.default_rng(17)
    kinds = []
    for rows, per in [(0, 0), (1, 0), (1, 1), (3, 2), (9, 3), (40, 5), (300, 4), (5000, 1)]:
        rp = np.arange(rows + 1, dtype=np.int32) * per
        col = np.sort(np.argsort(rng.random((rows, max(rows, 1))), axis=1)[:, :per], axis=1) if rows < 1000 else \
            rng.integers(0, rows, (rows, 1))
        val = rng.uniform(-1, 1, rows * per).astype(np.float32).astype(np.float64)
        kinds.append(hsmu.HostMatrix(rows, rows, rp, col.astype(np.int32).ravel(), val))
    order = np.concatenate([rng.integers(0, 7, 3000), [7], np.zeros(6000, np.int64), rng.integers(0, 6, 1500),
                            np.ones(5000, np.int64), [4, 7, 0, 0]])
    print(f"[gpu-case] stack of {len(order)} instances, same {same} {opts}", flush=True)
    fp32 = "precision" in opts
    dev = [ctx.matrix(k, fp32) for k in kinds]
    dev2 = dev if same else [ctx.matrix(k, fp32) for k in kinds]
    Cs, _ = ctx.spgemm_batched_device([dev[k] for k in order], [dev2[k] for k in order], hsmu.default_opts(**opts))
    refs = [oracle.spgemm(k, k) for k in kinds]
    try:
        for i, k in enumerate(order):
            ref = refs[k]
            assert Cs[i].nnz == ref.rowptr[-1]
            if k < 2 and i % 50:  # (no entries: a sample)
                continue
            C = ctx.fetch(Cs[i])
            assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
            bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
            assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)
    finally:
        ctx.free_batch(Cs)
