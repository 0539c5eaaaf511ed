"""A transposed copy that starts on no 16-byte boundary (packed into a larger buffer by the caller): the operand that would be
read in place next to it goes through its own transposed copy instead, as any other misaligned operand does."""
import pytest
import torch

from nanotron_amd.fp8.dtypes import DTypes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1, 8, 16])
def test_weight_gradient_with_a_packed_copy(offset):
    from nanotron_amd.fp8 import FP8Tensor
    from nanotron_amd.fp8.kernel import fp8_matmul_kernel

    g = torch.Generator(device="cuda").manual_seed(offset)
    x = FP8Tensor(torch.randn(512, 272, generator=g, device="cuda"), DTypes.FP8E4M3)
    dy = FP8Tensor(torch.randn(512, 320, generator=g, device="cuda"), DTypes.FP8E5M2, with_transpose=True)
    want = fp8_matmul_kernel(x, False, dy, True, True)
    copy = dy.transposed()
    packed = torch.empty(offset + copy.numel(), dtype=torch.uint8, device="cuda")[offset:].view(copy.shape)
    packed.copy_(copy.as_subclass(torch.Tensor))
    dy._transposed = torch.Tensor._make_subclass(FP8Tensor, packed)
    dy._transposed.fp8_meta = dy.fp8_meta
    got = fp8_matmul_kernel(x, False, dy, True, True)
    # (the aligned forms run the same instructions in the same order; others sum in fp32 throughout: 512 products)
    assert float((got - want).norm() / want.norm()) <= (0.0 if offset % 16 == 0 else 6e-5)
