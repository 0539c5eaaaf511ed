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
