"""Wide rows with kept directories, flat and two-level, where the windows' lists cannot be had: a
workgroup per row.  An allocation-free call of so many small rows that their lists (64 bytes a row)
exceed what its 256 MiB leave, against the CPU oracle."""
import ctypes as C

import numpy as np
import pytest

import hsmu
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["flat", "two-level"])
@pytest.mark.parametrize("fp32", [False, True])
def test_a_workgroup_per_row(ctx, form, fp32):
    rng = np.random.default_rng(51)
    if form == "flat":  # spans of a tile: 92 bytes of workspace a row besides the lists
        M, N, opts = 2000000, 64, dict(force_global=1)
        col = np.sort(np.argsort(rng.random((500, N)), axis=1)[:, :3], axis=1)
    else:  # two tiles far apart: directories of two coarse words and two tiles, 128 bytes
        M, N, opts = 1450000, 64 * 120, dict(lds_row_max=96)
        col = np.stack([rng.integers(0, 1000, 500), rng.integers(N - 1000, N, 500)], 1)
    K, per = col.shape
    B = hsmu.HostMatrix(K, N, (np.arange(K + 1) * per).astype(np.int32), col.astype(np.int32).ravel(),
                        rng.uniform(-1, 1, K * per).astype(np.float32).astype(np.float64))
    A = hsmu.HostMatrix(M, K, np.arange(M + 1, dtype=np.int32), rng.integers(0, K, M).astype(np.int32),
                        rng.uniform(-1, 1, M).astype(np.float32).astype(np.float64))
    ref = oracle.spgemm(A, B)
    n = int(ref.rowptr[-1])
    print(f"[gpu-case] a workgroup per row, {form} directories, fp32 {fp32}", flush=True)
    fn = hsmu.lib.hsmu_spgemm_noalloc
    fn.restype = C.c_int
    fn.argtypes = [C.c_void_p, C.POINTER(hsmu.Csr), C.POINTER(hsmu.Csr), C.POINTER(hsmu.Csr), C.c_int64,
                   C.POINTER(hsmu.Opts), C.POINTER(hsmu.Stats)]
    vt = np.float32 if fp32 else np.float64
    dA, dB = ctx.matrix(A, fp32), ctx.matrix(B, fp32)
    out = [ctx.upload(np.zeros(M + 1, np.int32)), ctx.upload(np.zeros(n, np.int32)), ctx.upload(np.zeros(n, vt))]
    o = hsmu.default_opts(precision=hsmu.HSMU_FP32_COMP if fp32 else hsmu.HSMU_FP64, **opts)
    c, st = hsmu.Csr(0, 0, 0, *out, 0, 0), hsmu.Stats()
    try:
        rc = fn(ctx.handle, C.byref(dA.csr), C.byref(dB.csr), C.byref(c), n, C.byref(o), C.byref(st))
        assert rc == hsmu.HSMU_OK, hsmu.lib.hsmu_last_error()
        assert st.to_dict()["num_bin_rows"][8] == M and c.nnz == n
        got = ctx.fetch(c)
        assert np.array_equal(np.asarray(got.rowptr, np.int64), ref.rowptr) and np.array_equal(got.col, ref.col)
        bound = 2.0 ** -23 * np.abs(ref.val) + 1e-10 * ref.absval if fp32 else 1e-12 * ref.absval
        assert np.all(np.abs(got.val.astype(np.float64) - ref.val) <= bound)
    finally:
        for p in out:
            ctx.dfree(p)
        dA.free()
        dB.free()
