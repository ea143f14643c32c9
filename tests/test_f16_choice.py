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


@pytest.mark.parametrize("m,k,n,want", [
    (3852, 672, 5984, "stream"),   # us: 52.8, 56.8 on 256 x 64 tiles
    (4589, 544, 7584, "stream"),   # 70.2 / 74.6
    (14468, 608, 3520, "stream"),  # 99 / 112
    (2140, 1376, 1056, "ring"),    # 22.7 / 26.5
    (1920, 2592, 1184, "ring"),    # 31.8 / 33.8
    (2181, 1664, 928, "ring"),     # 23.7 / 27.3
    (4173, 1536, 6144, "wide"),
    (4173, 6144, 1536, "stream"),
    (2048, 4096, 14336, "wide"),
    (4096, 4096, 1024, "wide"),
])
def test_predicted_tiles(m, k, n, want):
    assert h.f16_rows_kernel(m, k, n)[0] == want


@pytest.mark.parametrize("m,k,n,slices,image", [
    (362, 7232, 1056, 8, True),   # us: image 26.8, fp32 rows 30.3
    (294, 6304, 96, 8, True),     # 17.7 / 18.6
    (500, 6144, 1536, 5, True),
    (1024, 5760, 640, 6, False),  # 29.1 / 26.7
    (2048, 4608, 512, 4, False),
])
def test_splitk_form(m, k, n, slices, image):
    """From 257 rows the split-K path's workspace holds the fp16 image only
    where that form runs."""
    mp = (m + 15) // 16 * 16
    need = slices * mp * n * 4 + (mp * k * 2 + 255) // 256 * 256 * image
    assert h.f16_workspace_bytes(m, k, n) == max(need, mp * k * 2)
