"""The native host calls refuse tensors in host memory: a kernel handed such an address would fault the GPU."""
import pytest
import torch

from nanotron_amd import _native as nt

F8 = torch.zeros(16, 16, dtype=torch.uint8)
X = torch.zeros(16, 16)
ONE = torch.ones(1)


@pytest.mark.parametrize("call", [
    lambda: nt.host.quantize(X, 0, 0, None, None, 0, False),
    lambda: nt.host.quantize_batch([(X, ONE, 1, 0, False)], 0),
    lambda: nt.host.cast(X, ONE, 0, False),
    lambda: nt.host.cast_with_scale(X, ONE, 0, False),
    lambda: nt.host.column_sum(X, 0),
    lambda: nt.host.dequantize(F8, 0, ONE, 0, False),
    lambda: nt.host.transpose(F8),
    lambda: nt.host.gemm(F8, 0, ONE, F8, 0, ONE, 0, None, False, None, False),
], ids=["quantize", "quantize_batch", "cast", "cast_with_scale", "column_sum", "dequantize", "transpose", "gemm"])
def test_host_memory_is_refused(call):
    with pytest.raises(AssertionError):
        call()
