"""GPU parity of the GEMM for a few rows (`gemm_few_kernel`) at the edges of its row blocks, of its 16 or 32 columns, of
the K-tiles that its eight waves take in turn (a short last one, a round that not all waves share) and of the rule that
sends a problem there.  Operands are small integers, so every sum is exact in fp32 and the result is compared bit for
bit; 16-bit outputs with the exact value rounded once."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(M, N, K):
    from nanotron_amd import _native as nt

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M * 7 + N + K)

    def operand(rows, dtype):
        v = torch.randint(-3, 4, (rows, K), generator=g, device=dev).float()
        return v, v.to(dtype).view(torch.uint8)

    one = torch.ones(1, device=dev)
    bias = torch.randint(-4, 5, (N,), generator=g, device=dev).float()
    base = torch.randint(-50, 51, (M, N), generator=g, device=dev).float()
    for fa, fb in [(nt.E4M3, nt.E4M3), (nt.E5M2, nt.E4M3)]:
        types = {nt.E4M3: torch.float8_e4m3fn, nt.E5M2: torch.float8_e5m2}
        (a, aq), (b, bq) = operand(M, types[fa]), operand(N, types[fb])
        ref = a @ b.t()
        print(f"M={M} N={N} K={K} formats {fa} {fb}", flush=True)
        for odt in (torch.float32, torch.bfloat16, torch.float16):
            code = nt.TORCH_TO_NT[odt]
            assert torch.equal(nt.host.gemm(aq, fa, one, bq, fb, one, code, None, False, None, False), ref.to(odt))
            assert torch.equal(nt.host.gemm(aq, fa, one, bq, fb, one, code, None, False, bias, False), (ref + bias).to(odt))
        out = base.clone()
        nt.host.gemm(aq, fa, one, bq, fb, one, nt.F32, out, False, None, False)
        assert torch.equal(out, ref + base)


@pytest.mark.parametrize("mn", [(1, 1), (3, 15), (16, 17), (15, 4096), (5, 4121), (16, 8177), (2, 8193)])
@pytest.mark.parametrize("K", [2032, 2048, 2064, 4112, 9216])
def test_sixteen_rows(mn, K):
    _check(*mn, K)


@pytest.mark.parametrize("mn", [(17, 1), (31, 2047), (32, 33), (32, 4097), (33, 40)])
@pytest.mark.parametrize("K", [6128, 6144, 6160, 9216])
def test_thirty_two_rows(mn, K):
    _check(*mn, K)
