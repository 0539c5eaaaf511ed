"""Flat and transposing quantisation at the edges of what one workgroup takes: spans of 16384 elements, 16-byte loads,
128-wide tiles whose rows start on lines or anywhere, and pointers that no wide load may use, against the oracle."""
import pytest
import torch

from nanotron_amd.fp8 import DelayedScaling, DTypes, FP8Tensor
from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu
SPAN = 16384
CUS = 256
FORMATS = {"e4m3": (DTypes.FP8E4M3, O.E4M3), "e5m2": (DTypes.FP8E5M2, O.E5M2)}


def _tensor(shape, dtype, seed, offset=0):
    g = torch.Generator().manual_seed(seed)
    n = 1
    for s in shape:
        n *= s
    x = torch.randn(n + offset, generator=g)
    x[torch.randint(0, n, (3,), generator=g)] = torch.tensor([float("nan"), 40.0, -0.0])
    return x.to(dtype)[offset:].reshape(shape)


def _check(x, fmt, transpose, offset=0):
    dt, of = FORMATS[fmt]
    dev = torch.empty(x.numel() + offset, dtype=x.dtype, device="cuda")[offset:].reshape(x.shape)
    dev.copy_(x)
    ref = O.quantise_current(x, of)
    q = FP8Tensor(dev, dt, with_transpose=transpose)
    assert torch.equal(q.as_subclass(torch.Tensor).cpu(), ref.q)
    if transpose:
        assert torch.equal(q.transposed().as_subclass(torch.Tensor).cpu(), ref.q.t().contiguous())
    # the same bytes with the held scale of a delayed role (amax, cast and bookkeeping in one pass)
    finite = torch.nan_to_num(x.float(), nan=1.0).to(x.dtype)
    state = DelayedScaling(dt, 4, 0, "cuda")
    dev.copy_(finite)
    FP8Tensor(dev, dt, state=state, with_transpose=transpose)   # first use
    assert state.initialised
    d = FP8Tensor(dev, dt, state=state, with_transpose=transpose)
    want = O.quantise_current(finite, of)
    assert torch.equal(d.as_subclass(torch.Tensor).cpu(), want.q)
    assert d.fp8_meta.amax.item() == finite.float().abs().max().item()
    if transpose:
        assert torch.equal(d.transposed().as_subclass(torch.Tensor).cpu(), want.q.t().contiguous())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [9, 1024 * 8, 1024 * 8 + 7, 66000, CUS * 4096 + 3, CUS * 8192, CUS * 8192 + 8, 4 * SPAN + 1, 5 * SPAN - 1, 7 * SPAN + 8 * 37 + 3, 2 * CUS * SPAN - 4, (2 * CUS + 1) * SPAN + 5])
def test_flat_spans(n, dtype):
    _check(_tensor((1, n), dtype, n), "e4m3" if n % 2 else "e5m2", False)


@pytest.mark.parametrize("offset", [1, 4])
def test_flat_misaligned(offset):
    _check(_tensor((1, 6 * SPAN + 77), torch.bfloat16, offset, offset), "e4m3", False, offset)


# 128-wide tiles need 160 (delayed step) or 224 (cast) of them; columns: whole lines, 16-byte rows, rows that start anywhere
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,cols", [(2048, 2048), (2045, 2112), (2050, 2056), (1999, 2049)])
def test_tiles(rows, cols, dtype):
    _check(_tensor((rows, cols), dtype, rows + cols), "e4m3" if rows % 2 else "e5m2", True)


@pytest.mark.parametrize("offset", [8, 3])
def test_tiles_off_the_line(offset):
    _check(_tensor((2048, 2048), torch.float32, offset, offset), "e4m3", True, offset)
