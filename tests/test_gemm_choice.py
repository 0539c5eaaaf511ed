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


@pytest.mark.parametrize("mn", [(3632, 1088), (1568, 2496), (5400, 704), (16500, 192)])   # 387 to 507 tiles of 128 x 64, up to 75 of 256
@pytest.mark.parametrize("out,copy,K,want", [
    (BF16, 0, 256, (256, 256, 2)), (BF16, 0, 512, (256, 256, 2)), (BF16, 0, 1536, (256, 256, 2)), (BF16, 0, 4096, (128, 64, 1)),
    (F32, 0, 256, (256, 256, 2)), (F32, 0, 1024, (128, 64, 1)), (F32, 0, 4096, (128, 64, 1)),
    (OUT_E4M3, 0, 256, (256, 256, 2)), (OUT_E4M3, 0, 1536, (256, 256, 2)), (OUT_E4M3, 0, 4096, (128, 64, 1)),
    (OUT_E4M3, 1, 256, (256, 256, 2)), (OUT_E4M3, 1, 3072, (256, 256, 2)),
])
def test_second_round_of_128_x_64_tiles(mn, out, copy, K, want):
    assert tiles((*mn, K, out, 0), copy=copy) == want


@pytest.mark.parametrize("layer,out,acc,want", [   # (tokens, in features, out features); us in the tiles wanted / others
    ((256, 256, 7760), BF16, False, (64, 64)),      # 20.4 / 128 x 64 27.4
    ((288, 256, 3840), BF16, False, (64, 64)),      # 9.4 / 128 x 64 12.6
    ((432, 256, 3824), F32, False, (64, 64)),       # 11.6 / 128 x 64 15.9
    ((256, 448, 4416), BF16, True, (64, 64)),       # 13.8 / 128 x 128 19.9
    ((768, 1056, 3184), BF16, True, (256, 256)),    # 22.9 / 128 x 128 28.3
    ((976, 1136, 3664), F32, True, (256, 256)),     # 28.2 / 128 x 128 34.0
    ((2304, 1520, 3584), BF16, False, (256, 256)),  # 40.3 / 128 x 128 44.1
    ((1280, 2560, 6912), BF16, False, (128, 128)),  # 62 / 256 x 256 82
])
def test_input_and_weight_gradient_in_one_launch(layer, out, acc, want):
    tokens, fin, fout = layer
    assert tiles((tokens, fin, fout, out, 1), (fout, fin, tokens, F32, 2, acc))[:2] == want


@pytest.mark.parametrize("a,b", [((3904, 256, 384, BF16, 0), (224, 352, 7152, BF16, 0)),       # 13.9 / 128 x 64 22.1
                                 ((1280, 768, 2016, BF16, 0), (160, 400, 3984, BF16, 0))])     # 10.3 / 128 x 64 14.3
def test_deep_tiles_beside_shallow_ones(a, b):
    assert tiles(a, b)[:2] == tiles(b, a)[:2] == (64, 64)


@pytest.mark.parametrize("cus", [1, 7, 64, 256, 304])
def test_any_list_on_any_gpu(cus):
    for a, b in [((304, 304, 256, F32, 2), (70000, 4096, 512, F32, 2, True)), ((272, 272, 8192, F32, 2), (272, 272, 256, F32, 2)),
                 ((100000, 8192, 256, F32, 2), (100000, 8192, 512, F32, 2))]:
        assert tiles(a, b, cus=cus) is not None and tiles(a, b, a, b, cus=cus) is not None


def test_what_other_kernels_serve():
    assert tiles((16, 4096, 4096, BF16, 0)) is None             # a few rows
    assert tiles((4096, 4096, 128, BF16, 0)) is None            # one K-tile, more tiles than the chip works on at once
    assert tiles((1021, 2304, 1021, BF16, 0)) is None           # K no multiple of 16
    assert tiles((1021, 2304, 1024, OUT_E4M3, 0)) is None       # fp8 output, rows that do not come in fours
