"""GEMMs with fp8 outputs whose last workgroup does the output role's bookkeeping: bytes, amax, history and scales equal the
fp32 GEMM followed by the fused delayed-scaling quantisation, bit for bit, for every kernel that serves a shape and over
steps in a row (the workspace is left zero)."""
import pytest
import torch

from nanotron_amd.fp8.dtypes import DTypes

pytestmark = pytest.mark.gpu

SHAPES = [
    (16, 16, 32), (200, 336, 272), (512, 512, 512),   # 64-wide tiles
    (2000, 2032, 768),                                # 128-wide
    (1124, 5120, 1024),                               # halves of 256-wide tiles, the last row of them empty
    (4096, 6144, 512),                                # whole tiles and a tail
    (1024, 2048, 144), (1056, 2048, 144),             # 512 tiles of 64 (one round, bookkeeping inside) and more
    (1072, 3600, 320),                                # 256- and 64-wide tiles at equal estimates
    (1024, 4096, 240), (1040, 4112, 240),             # few K-tiles, both sides of the line to gemm_nt_kernel
    (1472, 1408, 77), (1500, 1500, 77),               # the same of tiles for any K (506 and 576)
    (64, 40, 77), (200, 300, 333),                    # K a multiple of nothing
    (66, 100, 128), (33, 18, 64),                     # rows and columns that do not come in words
]


@pytest.mark.parametrize("mnk", SHAPES)
@pytest.mark.parametrize("fmt", [DTypes.FP8E4M3, DTypes.FP8E5M2])
def test_bookkeeping_in_the_gemm(mnk, fmt):
    from nanotron_amd.fp8 import DelayedScaling, FP8Tensor
    from nanotron_amd.fp8.kernel import fp8_matmul_kernel

    M, N, K = mnk
    g = torch.Generator(device="cuda").manual_seed(M + K)
    one, two = (DelayedScaling(fmt, 3, 0, "cuda") for _ in range(2))
    for step in range(4):
        x = FP8Tensor(torch.randn(M, K, generator=g, device="cuda") * (1 + step), DTypes.FP8E4M3)
        w = FP8Tensor(torch.randn(N, K, generator=g, device="cuda"), DTypes.FP8E4M3)
        print(f"{mnk} {fmt} step {step}", flush=True)
        got = fp8_matmul_kernel(w, True, x, False, False, out_dtype=fmt, out_state=one)
        want = FP8Tensor(fp8_matmul_kernel(w, True, x, False, False), fmt, state=two)
        assert one.initialised and two.initialised   # (from the second step on the epilogue casts)
        assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor))
        assert torch.equal(one._buf, two._buf)
        assert got.fp8_meta.amax.item() == want.fp8_meta.amax.item() and got.fp8_meta.scale.item() == want.fp8_meta.scale.item()


# rows and columns that end inside a tile, some of them after one element: (M, N, K)
RAGGED = [
    (1, 1, 7), (1, 16, 515), (20, 48, 33), (130, 129, 77),          # K a multiple of nothing
    (4, 16, 32), (20, 48, 64), (100, 80, 272), (132, 144, 128),     # 64-wide tiles
    (2052, 2064, 768),                                              # 128-wide
    (1124, 5136, 1024),                                             # halves of 256-wide tiles
    (4100, 6160, 512),                                              # whole tiles and a tail
    (1, 1, 16), (66, 100, 128), (33, 18, 64),                       # rows and columns that do not come in words
]


def _held(fmt):
    """Two delayed-scaling states that hold the same scale (so that the epilogue casts)."""
    from nanotron_amd.fp8 import DelayedScaling, FP8Tensor

    states = [DelayedScaling(fmt, 3, 0, "cuda") for _ in range(2)]
    for s in states:
        FP8Tensor(torch.full((16,), 3.0, device="cuda"), fmt, state=s)
        assert s.initialised
    return states


def _same(got, want, one, two, amax):
    assert got.fp8_meta.amax.item() == want.fp8_meta.amax.item() == amax
    assert torch.equal(one._buf, two._buf)
    assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor))


@pytest.mark.parametrize("mnk", RAGGED)
def test_bias_of_padding_rows_stays_out_of_the_amax(mnk):
    """Every result is K + (1/8 - K): a row that is not there would count as |1/8 - K|."""
    from nanotron_amd.fp8 import FP8Tensor
    from nanotron_amd.fp8.kernel import fp8_matmul_kernel

    M, N, K = mnk
    print(f"{mnk}", flush=True)
    fmt = DTypes.FP8E4M3
    one, two = _held(fmt)
    x, w = (FP8Tensor(torch.ones(r, K, device="cuda"), DTypes.FP8E4M3) for r in (M, N))
    bias = torch.full((N,), 0.125 - K, device="cuda")
    got = fp8_matmul_kernel(w, True, x, False, False, out_dtype=fmt, out_state=one, bias=bias)
    want = FP8Tensor(fp8_matmul_kernel(w, True, x, False, False, bias=bias), fmt, state=two)
    _same(got, want, one, two, 0.125)


@pytest.mark.parametrize("infinite", ["x", "w"])
@pytest.mark.parametrize("mnk,plain_w", [(s, True) for s in RAGGED] + [((132, 144, 256), False), ((2052, 2064, 768), False)])
def test_infinite_operand_against_padding_stays_out_of_the_amax(mnk, plain_w, infinite):
    """An infinite code makes one row or column of the result infinite; against the zeros of padding it makes NaN, which
    must not become the amax."""
    from nanotron_amd.fp8 import FP8Tensor
    from nanotron_amd.fp8.kernel import fp8_matmul_kernel

    M, N, K = mnk
    print(f"{mnk} {plain_w} {infinite}", flush=True)
    fmt = DTypes.FP8E5M2
    one, two = _held(fmt)
    x, w = (FP8Tensor(torch.ones(s, device="cuda"), DTypes.FP8E5M2) for s in ((M, K), (N, K) if plain_w else (K, N)))
    (x if infinite == "x" else w).as_subclass(torch.Tensor)[0, 0] = 0x7c   # +Inf in e5m2
    got = fp8_matmul_kernel(w, plain_w, x, False, False, out_dtype=fmt, out_state=one)
    want = FP8Tensor(fp8_matmul_kernel(w, plain_w, x, False, False), fmt, state=two)
    _same(got, want, one, two, float("inf"))
