"""int4 tiles of 256 x 256 against 128 x 256 (wq_gemm_plan.cpp), asked on problems whose builds were timed on an MI355X, canonical weights from memory."""
import pytest

from tests.test_gemm_plan_cpu import ask  # noqa: F401

TILE_256X256 = 3

# (M, N, K, us in 128 x 256 tiles, us in 256 x 256)
TIMED = [
    (1087, 12288, 3840, 101.0, 107.2), (800, 14336, 9472, 219.2, 233.2), (861, 15104, 9472, 233.2, 245.2), (1670, 29184, 3072, 300.4, 328.2),  # rounds that are not full
    (1720, 28288, 7680, 717.0, 778.4), (1766, 31616, 4096, 408.2, 430.8),
    (1400, 8933, 1280, 46.7, 64.1), (1945, 6461, 3072, 88.9, 104.8), (1465, 21309, 1536, 117.3, 148.3), (1708, 8357, 4352, 126.4, 141.4),  # odd N
    (1143, 12837, 5120, 148.7, 170.8), (474, 28959, 5376, 152.0, 165.6), (1831, 31637, 4096, 484.1, 547.7),
    (2048, 22016, 4096, 335.8, 327.5), (406, 25600, 6656, 159.6, 155.7), (1951, 30080, 5120, 566.0, 553.7), (467, 29312, 2304, 69.5, 67.9)]


@pytest.mark.parametrize("tiled", [0, 1])
@pytest.mark.parametrize("m,n,k,us_128,us_256", TIMED)
def test_256x256_tiles_where_they_are_ahead(ask, m, n, k, us_128, us_256, tiled):  # noqa: F811
    assert (ask(4, m, n, k, tiled)[0] == TILE_256X256) == (us_256 < us_128)
