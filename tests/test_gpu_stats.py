"""Statistics that stay the same per row whatever the number of rows."""
import pytest

import hsmu

pytestmark = pytest.mark.gpu


def test_lds_of_rows_that_share_a_wave(ctx):
    """lds_launched is the LDS all row groups ask for: the same per row on a small grid and on
    one of more groups than there are workgroups (their 8-lane rows differ only at the rim)."""
    per_row = []
    for n in (300, 900):
        A = hsmu.gen_laplace2d(n)
        print(f"[gpu-case] lds_launched of a {n} x {n} grid", flush=True)
        _, st = ctx.spgemm(A, A)
        assert st["num_bin_rows"][0] == A.M
        per_row.append(st["lds_launched"] / A.M)
        assert 0 < st["lds_use"] <= 1
        assert st["lds_use"] * st["lds_launched"] == pytest.approx(12.0 * st["nnz_c"], rel=1e-12)
    assert per_row[1] == pytest.approx(per_row[0], rel=1e-3)
