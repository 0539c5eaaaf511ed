"""GPU parity of the 128- and 64-wide GEMM tiles (`gemm_mid_kernel`) at the edges of their tiles and of their pipeline
(one to six K-tiles of 128 bytes, the last one short), for every operand layout and output type.  Operands are small
integers, so every sum is exact in fp32 and the result is compared bit for bit; 16-bit outputs with the exact value
rounded once."""
import pytest
import torch

from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu

SMALL = [(1, 1), (16, 130), (63, 65), (64, 64), (100, 36), (129, 200)]     # 64-wide tiles
LARGE = [(1900, 1936), (2048, 2033)]                                       # 128-wide: one tile per CU at most
KS = [16, 128, 144, 272, 400, 640]


def _check(M, N, K, form, odt, acc=False, bias=False):
    from nanotron_amd import _native as nt

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M * 7 + N + K)

    def operand(rows):
        v = torch.randint(-3, 4, (rows, K), generator=g, device=dev).float()
        return v, v.to(torch.float8_e4m3fn).view(torch.uint8)

    (a, aq), (b, bq) = operand(M), operand(N)
    bt, at = form != "plain", form == "both"
    if bt:
        bq = bq.t().contiguous()
    if at:
        aq = aq.t().contiguous()
    one = torch.ones(1, device=dev)
    ref = a @ b.t()
    bv = torch.randint(-4, 5, (N,), generator=g, device=dev).float() if bias else None
    base = torch.randint(-50, 51, (M, N), generator=g, device=dev).float() if acc else None
    out = base.clone() if acc else torch.full((M, N), 7.0, dtype=odt, device=dev)
    print(f"M={M} N={N} K={K} {form} {odt} acc={acc} bias={bias}", flush=True)
    got = nt.host.gemm(aq, nt.E4M3, one, bq, nt.E4M3, one, nt.TORCH_TO_NT[odt], out if acc else None, bt, bv, at)
    if bias:
        ref = ref + bv
    if acc:
        ref = ref + base
    assert torch.equal(got, ref.to(odt))


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("mn", SMALL + LARGE)
def test_plain_operands(mn, K):
    _check(*mn, K, "plain", torch.float32)
    _check(*mn, K, "plain", torch.bfloat16, bias=True)
    _check(*mn, K, "plain", torch.float32, acc=True)


@pytest.mark.parametrize("K", [k for k in KS if k >= 256])
@pytest.mark.parametrize("mn", [(144, 144), (208, 272), (1904, 1936)])
@pytest.mark.parametrize("form", ["b", "both"])
def test_transposed_operands(mn, K, form):
    _check(*mn, K, form, torch.float32)
    _check(*mn, K, form, torch.float16)
    _check(*mn, K, form, torch.float32, acc=True)


def test_problems_of_different_layout_and_depth_in_one_call():
    from nanotron_amd import _native as nt

    dev = torch.device("cuda", 0)
    one = torch.ones(1, device=dev)
    g = torch.Generator(device=dev).manual_seed(5)
    for T, fin, fout in [(256, 272, 528), (1024, 1040, 512)]:   # 64-wide, 128-wide
        dy = torch.randint(-3, 4, (T, fout), generator=g, device=dev).float()
        x, w = (torch.randint(-3, 4, s, generator=g, device=dev).float() for s in ((T, fin), (fout, fin)))
        q = [t.to(torch.float8_e4m3fn).view(torch.uint8) for t in (dy, x, w)]
        dx, dw = nt.host.gemm_batch([(q[0], 0, one, q[2], 0, one, nt.BF16, None, True, None, False),
                                     (q[0], 0, one, q[1], 0, one, nt.F32, None, True, None, True)])
        assert torch.equal(dx, (dy @ w).to(torch.bfloat16)) and torch.equal(dw, dy.t() @ x)


@pytest.mark.parametrize("K", [16, 128, 240, 256])
@pytest.mark.parametrize("mn", [(1024, 4096), (1040, 4100), (1009, 1008), (1025, 1008), (1030, 1001), (2100, 2130)])
def test_large_results_of_few_k_tiles(mn, K):
    """Both sides of the lines beyond which a launch of fewer than two K-tiles goes to gemm_nt_kernel."""
    _check(*mn, K, "plain", torch.float32)
    _check(*mn, K, "plain", torch.float32, acc=True)
    _check(*mn, K, "plain", torch.bfloat16, bias=True)
    _check(*mn, K, "plain", torch.float16)
