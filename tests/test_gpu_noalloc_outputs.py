"""An allocation-free call that fails leaves the caller's int32 row pointers as they were."""
import ctypes as C

import numpy as np
import pytest

import hsmu
import oracle

pytestmark = pytest.mark.gpu


def test_failed_call_keeps_row_pointers(ctx):
    fn = hsmu.lib.hsmu_spgemm_noalloc
    fn.restype = C.c_int
    fn.argtypes = [C.c_void_p, C.POINTER(hsmu.Csr), C.POINTER(hsmu.Csr), C.POINTER(hsmu.Csr), C.c_int64,
                   C.POINTER(hsmu.Opts), C.POINTER(hsmu.Stats)]
    A = hsmu.gen_random(500, 300, 9, 1)
    B = hsmu.gen_random(300, 4000, 20, 2)
    ref = oracle.spgemm(A, B)
    n = int(ref.rowptr[-1])
    dA, dB = ctx.matrix(A), ctx.matrix(B)
    mark = np.full(A.M + 1, -77, np.int32)
    rp, col, val = ctx.upload(mark), ctx.upload(np.zeros(n, np.int32)), ctx.upload(np.zeros(n))
    o, st = hsmu.default_opts(), hsmu.Stats()
    try:
        for cap in (n - 1, n):
            print(f"[gpu-case] noalloc with room for {cap} of {n}", flush=True)
            c = hsmu.Csr(0, 0, 0, rp, col, val, 0, 0)
            rc = fn(ctx.handle, C.byref(dA.csr), C.byref(dB.csr), C.byref(c), cap, C.byref(o), C.byref(st))
            got = ctx.download(rp, A.M + 1, np.int32)
            assert rc == (hsmu.HSMU_OK if cap == n else hsmu.HSMU_ERR_NOMEM)
            assert np.array_equal(got, ref.rowptr if cap == n else mark)
        assert np.array_equal(ctx.download(col, n, np.int32), ref.col)
    finally:
        for p in (rp, col, val):
            ctx.dfree(p)
        dA.free()
        dB.free()
