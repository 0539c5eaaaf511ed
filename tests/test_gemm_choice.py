"""Tile sizes of GEMM launches on a GPU of 256 CUs, at shapes that were timed in every one of them."""
import pytest
from tile_choice import BF16, F32, OUT_E4M3, tiles


@pytest.mark.parametrize("problem,want", [
    ((1024, 1024, 1024, BF16, 0), (64, 64, 1)),       # us in 256- / 128- / 64-wide tiles 10.1 / 7.5 / 4.8
    ((2048, 1024, 4096, BF16, 0), (128, 64, 1)),      # 128 x 128 / 128 x 64 / 64 x 64: 15.6 / 12.9 / 15.2
    ((2048, 2048, 2048, BF16, 0), (128, 128, 1)),     # 16.7 / 11.8 / 16.9
    ((2048, 2048, 2048, F32, 2), (128, 128, 1)),      # 19.6 / 12.6 / 24.3
    ((2048, 4096, 4096, BF16, 0), (256, 256, 2)),     # 32.5 / 40.4 / 55.8: 128 tiles, in halves
    ((4096, 4096, 4096, BF16, 0), (256, 256, 1)),     # 51.9 / 73.5 / 101
    ((4400, 3900, 272, F32, 0), (256, 256, 8)),
])
def test_one_problem(problem, want):
    assert tiles(problem) == want


@pytest.mark.parametrize("mn", [(2656, 3072), (1888, 4352), (2688, 2864)])   # 132 to 136 tiles of 256, two rounds of 128-wide ones
@pytest.mark.parametrize("K", [768, 1024, 1152, 4096])
@pytest.mark.parametrize("out,form", [(BF16, 0), (F32, 0), (BF16, 1), (F32, 2)])
def test_two_rounds_of_128_wide_tiles(mn, K, out, form):
    assert tiles((*mn, K, out, form)) == (128, 128, 1)


@pytest.mark.parametrize("mn", [(2560, 3328), (2400, 3840), (3584, 2560), (3840, 4352)])   # 130 to 255 tiles of 256, more rounds of 128-wide ones
@pytest.mark.parametrize("K", [1024, 4096, 5120, 8192])
@pytest.mark.parametrize("out,form", [(BF16, 0), (F32, 0), (BF16, 1), (F32, 2)])
def test_part_of_the_chip_in_256_wide_tiles(mn, K, out, form):
    assert tiles((*mn, K, out, form)) == (256, 256, 1)


def test_what_other_kernels_serve():
    assert tiles((16, 4096, 4096, BF16, 0)) is None             # a few rows
    assert tiles((4096, 4096, 128, BF16, 0)) is None            # one K-tile, more tiles than the chip works on at once
    assert tiles((1021, 2304, 1021, BF16, 0)) is None           # K no multiple of 16
    assert tiles((1021, 2304, 1024, OUT_E4M3, 0)) is None       # fp8 output, rows that do not come in fours
