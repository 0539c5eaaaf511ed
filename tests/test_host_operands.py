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


class _OnTheGpu:
    """Stand-ins for tensors on a GPU (they have no memory: a call that reached for an address would raise something
    else than the refusal that is asked for)."""

    def __getitem__(self, _):
        from torch._subclasses.fake_tensor import FakeTensorMode

        with FakeTensorMode():
            return (torch.empty(16, 16, dtype=torch.uint8, device="cuda:0"), torch.empty(16, 16, device="cuda:0"),
                    torch.empty(1, device="cuda:0"), torch.empty(2, device="cuda:0"))


@pytest.mark.parametrize("bad", [torch.ones(3), "fp64", "empty"], ids=["host memory", "fp64", "no value"])
@pytest.mark.parametrize("call", [
    lambda f8, x, one, st, s: nt.host.quantize(x, 0, 0, s, None, 1, False),
    lambda f8, x, one, st, s: nt.host.quantize(x, 0, 0, st, s, 1, False),
    lambda f8, x, one, st, s: nt.host.quantize_batch([(x, s, 1, 0, False)], 0),
    lambda f8, x, one, st, s: nt.host.cast(x, s, 0, False),
    lambda f8, x, one, st, s: nt.host.cast_with_scale(x, s, 0, False),
    lambda f8, x, one, st, s: nt.host.dequantize(f8, 0, s, 0, False),
    lambda f8, x, one, st, s: nt.host.gemm(f8, 0, s, f8, 0, one, 0, None, False, None, False),
    lambda f8, x, one, st, s: nt.host.gemm(f8, 0, one, f8, 0, s, 0, None, False, None, False),
    lambda f8, x, one, st, s: nt.host.gemm_batch([(f8, 0, one, f8, 0, s, 0, None, False, None, False)]),
    lambda f8, x, one, st, s: nt.host.gemm_fp8(f8, 0, one, f8, 0, one, 3, None, False, None, False, s, 1, 0, False),
], ids=["quantize state", "quantize flag", "quantize_batch state", "cast", "cast_with_scale", "dequantize", "gemm a", "gemm b", "gemm_batch",
        "gemm_fp8 state"])
def test_scales_that_a_kernel_must_not_read_are_refused(call, bad):
    from torch._subclasses.fake_tensor import FakeTensorMode

    f8, x, one, state = _OnTheGpu()[0]
    if isinstance(bad, str):
        with FakeTensorMode():
            bad = torch.empty(0 if bad == "empty" else 3, dtype=torch.float64 if bad == "fp64" else torch.float32, device="cuda:0")
    with pytest.raises(AssertionError, match="scale"):
        call(f8, x, one, state, bad)


@pytest.mark.parametrize("call", [
    lambda x, one: nt.host.dequantize(x, 0, one, 0, False),
    lambda x, one: nt.host.transpose(x),
    lambda x, one: nt.host.gemm(x, 0, one, x, 0, one, 0, None, False, None, False),
], ids=["dequantize", "transpose", "gemm"])
def test_operands_that_are_no_fp8_codes_are_refused(call):
    _, x, one, _ = _OnTheGpu()[0]
    with pytest.raises(AssertionError, match="one byte"):
        call(x, one)
