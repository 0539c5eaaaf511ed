"""Edges of the tiles that leave a GEMM in whole lines (256 wide and halves of them, 128 x 64 and 64 wide), rows exchanged between lanes: every column remainder (lines, 64-byte pieces, 16-byte
chunks, none of them), row remainders of the 8 rows a store covers, the widest output, and nothing written around D.
Operands are small integers, so every sum is exact in fp32 and results are compared bit for bit."""
import ctypes

import pytest
import torch
from tile_choice import tiles

pytestmark = pytest.mark.gpu

SMALL = [(57, 32), (64, 48), (72, 36), (9, 8), (65, 130), (200, 96)]                            # 64-wide tiles
NARROW = [(2048, 1024), (1921, 1024), (2048, 961), (1935, 1000), (2045, 964)]                     # 128 x 64 tiles: one round of workgroups
TAILS = [(4400, 3900), (4361, 4100), (4352, 3856), (4097, 4352)]   # a round of 256-wide tiles and a few more, computed in quarters or eighths
HALVES = [(2301, 2064), (2303, 2080), (2297, 2548), (4091, 5904)]   # 81 or 90 of them, or 128 behind a full round: in halves
LARGE = [(4088, 4096), (4081, 4112), (4095, 4104), (3849, 4100), (4097, 3842), (2560, 3584)]     # 256-wide tiles


def _reaches(want, *problems, **kw):
    """The launch is in that tile size (256-wide: with its last round in that many parts)."""
    got = tiles(*problems, cus=torch.cuda.get_device_properties(0).multi_processor_count, **kw)
    assert got == ((*want, 1) if len(want) == 2 else want)


def _check(M, N, K, odt, acc, form="plain", full=True, tile=None):
    from nanotron_amd import _native as nt

    if tile is not None:
        _reaches(tile, (M, N, K, nt.TORCH_TO_NT[odt], ("plain", "b", "both").index(form), acc))
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M * 5 + N)
    a, b = (torch.randint(-2, 3, (r, K), generator=g, device=dev, dtype=torch.int8) for r in (M, N))
    aq, bq = (t.to(torch.float8_e4m3fn).view(torch.uint8) for t in (a, b))
    if form != "plain":
        bq = bq.t().contiguous()
    if form == "both":
        aq = aq.t().contiguous()
    guard = 64
    out = torch.full((guard + M * N + guard,), 9.0, dtype=odt, device=dev)
    one = torch.ones(1, device=dev)
    d = nt.GemmDesc(A=aq.data_ptr(), scale_a=one.data_ptr(), B=bq.data_ptr(), scale_b=one.data_ptr(),
                    D=out.data_ptr() + guard * out.element_size(), M=M, N=N, K=K, fmt_a=nt.E4M3, fmt_b=nt.E4M3,
                    d_dtype=nt.TORCH_TO_NT[odt], accumulate=int(acc), b_transposed=int(form != "plain"), a_transposed=int(form == "both"))
    print(f"M={M} N={N} K={K} {odt} acc={acc} {form}", flush=True)
    st = torch.cuda.current_stream().cuda_stream
    assert nt._lib.ntfp8_gemm_batch(ctypes.byref(d), 1, st) == 0
    assert bool((out[:guard] == 9.0).all()) and bool((out[guard + M * N:] == 9.0).all())
    got = out[guard:guard + M * N].view(M, N)
    cols = slice(0, N) if full else torch.cat([torch.arange(0, 300), torch.arange(N // 2, N // 2 + 300), torch.arange(N - 300, N)]).to(dev)
    want = a.float() @ b[cols].float().t() + (9.0 if acc else 0.0)
    assert torch.equal(got[:, cols], want.to(odt))


@pytest.mark.parametrize("mn", SMALL + NARROW + TAILS + LARGE)
@pytest.mark.parametrize("odt,acc", [(torch.float32, False), (torch.float32, True), (torch.bfloat16, False)])
def test_every_remainder(mn, odt, acc):
    _check(*mn, 272, odt, acc, tile=(64, 64) if mn in SMALL else (128, 64) if mn in NARROW else None)


@pytest.mark.parametrize("mn", HALVES)
@pytest.mark.parametrize("form", ["plain", "b"])
@pytest.mark.parametrize("odt,acc", [(torch.float32, False), (torch.float32, True), (torch.bfloat16, False)])
def test_every_remainder_of_halves(mn, form, odt, acc):
    if form == "plain" or mn[1] % 16 == 0:
        _check(*mn, 272, odt, acc, form, tile=(256, 256, 2))


@pytest.mark.parametrize("mn", [(2288, 2064), (2304, 2576), (4080, 5904)])
@pytest.mark.parametrize("acc", [False, True])
def test_transposed_operands_of_halves(mn, acc):
    _check(*mn, 272, torch.float32, acc, "both", tile=(256, 256, 2))


@pytest.mark.parametrize("mn", [(144, 144), (4096, 4112), (4112, 3856), (2048, 1024), (1936, 976), (2032, 1008),
                                (4400, 3904), (4368, 4112)])
@pytest.mark.parametrize("acc", [False, True])
def test_transposed_operands(mn, acc):
    _check(*mn, 272, torch.float32, acc, "both")


@pytest.mark.parametrize("mn", NARROW)
@pytest.mark.parametrize("K", [256, 400, 528, 656])
def test_narrow_tiles_of_two_and_more_k_tiles(mn, K):
    _check(*mn, K, torch.float32, False, tile=(128, 64))
    if mn[1] % 16 == 0:
        _check(*mn, K, torch.bfloat16, False, "b", tile=(128, 64))


@pytest.mark.parametrize("mn", [(2048, 512), (1935, 500), (1000, 961)])
@pytest.mark.parametrize("K", [16, 128])
@pytest.mark.parametrize("odt,acc", [(torch.float32, False), (torch.float32, True), (torch.bfloat16, False)])
def test_narrow_tiles_of_one_k_tile(mn, K, odt, acc):
    """One K-tile alone goes to other kernels; beside a deeper problem in the same launch it does not."""
    from nanotron_amd import _native as nt

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(K + mn[1])
    one = torch.ones(1, device=dev)
    _reaches((128, 64), (2048, 512, 1040, nt.TORCH_TO_NT[odt], 0), (*mn, K, nt.TORCH_TO_NT[odt], 0, acc))
    print(f"{mn} K={K} {odt} acc={acc}", flush=True)
    probs, wants = [], []
    for (M, N), k in (((2048, 512), 1040), (mn, K)):
        a, b = (torch.randint(-2, 3, (r, k), generator=g, device=dev).float() for r in (M, N))
        out = torch.full((M, N), 9.0, device=dev) if acc and k == K else None
        probs.append((a.to(torch.float8_e4m3fn).view(torch.uint8), nt.E4M3, one, b.to(torch.float8_e4m3fn).view(torch.uint8), nt.E4M3, one,
                      nt.TORCH_TO_NT[odt], out, False, None, False))
        wants.append((a @ b.t() + (0.0 if out is None else 9.0)).to(odt))
    for got, want in zip(nt.host.gemm_batch(probs), wants):
        assert torch.equal(got, want)


@pytest.mark.parametrize("mn", [(2048, 1024), (1924, 976), (2044, 1008), (4404, 3904), (4364, 4112)])
@pytest.mark.parametrize("form", ["plain", "b"])
def test_fp8_outputs(mn, form):
    from nanotron_amd import _native as nt

    (M, N), K = mn, 272
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + N)
    a, b = (torch.randint(-2, 3, (r, K), generator=g, device=dev).float() for r in (M, N))
    aq, bq = (t.to(torch.float8_e4m3fn).view(torch.uint8) for t in (a, b if form == "plain" else b.t().contiguous()))
    one, state = torch.ones(1, device=dev), torch.tensor([0.25, 0.0], device=dev)
    print(f"{mn} {form}", flush=True)
    y, y_t, amax, scale = nt.host.gemm_fp8(aq, nt.E4M3, one, bq, nt.E4M3, one, nt.OUT_E4M3, None, form == "b", None, False, state, 1, 0, True)
    r = a @ b.t()
    want = (r * 0.25).to(torch.float8_e4m3fn).view(torch.uint8)
    assert torch.equal(y, want) and torch.equal(y_t, want.t()) and float(amax) == float(r.abs().max()) and float(scale) == 0.25


@pytest.mark.parametrize("odt", [torch.float32, torch.bfloat16])
def test_more_columns_than_32_bit_offsets_reach(odt):
    _check(24, (1 << 22) + 16, 272, odt, False, full=False)
    _check(24, (1 << 22) - 16, 272, odt, False, full=False)
