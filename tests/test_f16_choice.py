"""Which kernel the F16 GEMM takes (host-side rules; on 256 CUs, also assumed
without a GPU).  Shapes are ones at which a rule was measured to be wrong, and
shapes on either side of each line."""
import pytest

import htp_ops as h


@pytest.mark.parametrize("m,k,n,want", [
    (200, 1184, 11392, ("stream", 256, 64)),  # 17.2 us; 23.9 on the ring kernel
    (212, 544, 14208, ("stream", 256, 64)),
    (193, 192, 8192, ("stream", 256, 64)),    # the least rows, k and n
    (231, 1728, 11232, ("stream", 256, 64)),
    (256, 2368, 8160, ("stream", 256, 64)),
    (256, 2400, 8192, ("wide", 256, 64)),
    (256, 4096, 14336, ("wide", 256, 64)),
    (240, 8192, 9216, ("wide", 256, 64)),
])
def test_one_row_of_256_row_tiles(m, k, n, want):
    """193-256 rows with columns for half of the CUs never take the ring kernel."""
    assert h.f16_rows_kernel(m, k, n) == want


@pytest.mark.parametrize("m,k,n", [(192, 1184, 11392), (200, 160, 11392), (200, 1184, 8064)])
def test_one_row_of_256_row_tiles_outside(m, k, n):
    assert h.f16_rows_kernel(m, k, n)[:2] != ("stream", 256)
