"""Stacking of a batch: instances that end within, at and across the workgroups' chunks of
4,096 entries and rows, empty ones among them, with A_i and B_i the same arrays and not,
against the CPU oracle."""
import numpy as np
import pytest

import hsmu
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("same", [True, False])
@pytest.mark.parametrize("fp32", [False, True])
def test_stack(ctx, same, fp32):
    rng = np.random.default_rng(3)
    print(f"[gpu-case] stack same {same} fp32 {fp32}", flush=True)
    hosts = []
    for rows, per in [(1, 1), (1, 0), (4096, 1), (2048, 2), (4095, 1), (1, 1), (9000, 3), (3, 1), (1365, 3), (5000, 0), (70, 60)]:
        rp = np.arange(rows + 1, dtype=np.int32) * per
        col = np.sort(np.argsort(rng.random((rows, max(rows, per) if rows < 100 else 64)), axis=1)[:, :per], axis=1)
        col = (col % rows if rows < 100 else (col + np.arange(rows)[:, None]) % rows)
        col = np.sort(col, axis=1).astype(np.int32).ravel()
        val = rng.uniform(-1, 1, rows * per).astype(np.float32).astype(np.float64)
        hosts.append(hsmu.HostMatrix(rows, rows, rp, col, val))
    o = hsmu.default_opts(precision=hsmu.HSMU_FP32_COMP if fp32 else hsmu.HSMU_FP64)
    dA = [ctx.matrix(X, fp32) for X in hosts]
    dB = dA if same else [ctx.matrix(X, fp32) for X in hosts]
    Cs, _ = ctx.spgemm_batched_device(dA, dB, o)
    got = [ctx.fetch(C) for C in Cs]
    ctx.free_batch(Cs)
    for X, C in zip(hosts, got):
        ref = oracle.spgemm(X, X)
        assert np.array_equal(np.asarray(C.rowptr, np.int64), ref.rowptr) and np.array_equal(C.col, ref.col)
        bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
        assert np.all(np.abs(C.val.astype(np.float64) - ref.val) <= bound)
