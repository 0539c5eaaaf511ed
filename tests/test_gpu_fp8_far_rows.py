"""fp8 outputs of almost 2^32 bytes: what the last tiles compute past the last row and the last column is dropped and lands
nowhere else in D or its transposed copy (its 32-bit offsets alone would begin again at the first rows).  Operands are small
integers, so every sum is exact in fp32 and results are compared bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,form", [(65300, 65760, "plain"), (65300, 65760, "b"),   # 256-wide tiles, rows and columns left over
                                      (260, 16519040, "plain")])                     # 128-wide ones
def test_last_tiles_stay_past_the_end(M, N, form):
    from nanotron_amd import _native as nt

    K = 256
    assert (M + 255) // 256 * 256 * N > 1 << 32 > M * N + 16
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(N)

    def operand(rows):   # +-1 and +-2 as e4m3 codes
        r = torch.randint(0, 4, (rows, K), generator=g, device=dev, dtype=torch.uint8)
        return 0x38 + (r & 1) * 8 + (r >> 1) * 128

    def widened(q):
        return q.view(torch.float8_e4m3fn).float()

    a, b = operand(M), operand(N)
    one, state = torch.ones(1, device=dev), torch.tensor([0.25, 0.0], device=dev)
    print(f"M={M} N={N} {form}", flush=True)
    y, y_t, amax, _ = nt.host.gemm_fp8(a, nt.E4M3, one, b if form == "plain" else b.t().contiguous(), nt.E4M3, one, nt.OUT_E4M3, None,
                                       form == "b", None, False, state, 1, 0, True)

    def block(rows, cols):   # of the result, and its largest value
        r = widened(a[rows]) @ widened(b[cols]).t()
        return (r * 0.25).to(torch.float8_e4m3fn).view(torch.uint8), float(r.abs().max())

    largest = 0.0
    step = (1 << 28) // N
    for rows in (slice(0, min(M, step)), slice(max(0, M - step), M)):
        for c in range(0, N, 1 << 20):
            cols = slice(c, min(N, c + (1 << 20)))
            want, top = block(rows, cols)
            assert torch.equal(y[rows, cols], want)
            largest = max(largest, top)
    for cols in (slice(0, 4096), slice(N - 4096, N)):
        for r in range(0, M, 1 << 14):
            rows = slice(r, min(M, r + (1 << 14)))
            want, top = block(rows, cols)
            assert torch.equal(y_t[cols, rows], want.t())
            largest = max(largest, top)
    assert float(amax) >= largest
