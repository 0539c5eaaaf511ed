"""GPU parity of the kernels that turn byte tiles around, at the edges of their 64- and 128-wide tiles and with rows
that start on no 16-byte boundary: exact."""
import pytest
import torch

from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu

# below one 128-wide tile per CU (64-wide tiles), and above it with remainders of every kind
SHAPES = [(1, 1), (1, 70), (67, 1), (63, 65), (64, 64), (129, 3), (200, 333), (128 * 16, 128 * 16), (128 * 16 + 1, 128 * 16 + 15),
          (128 * 16 + 14, 128 * 17 + 7),
          # one element per thread up to 131072 (delayed step) and 196608 (cast) elements, 64-wide tiles beyond
          (512, 256), (257, 511), (384, 512), (131, 1501), (449, 515), (1021, 703)]


@pytest.mark.parametrize("shape", SHAPES)
def test_transpose_of_bytes(shape):
    from nanotron_amd import _native as nt

    dev = torch.device("cuda", 0)
    rows, cols = shape
    for shift in (0, 1, 4):
        src = torch.randint(0, 256, (rows * cols + shift,), dtype=torch.uint8, device=dev)[shift:].view(rows, cols)
        store = torch.full((rows * cols + shift + 16,), 7, dtype=torch.uint8, device=dev)
        print(f"transpose {shape} shift {shift}", flush=True)
        nt.check(nt.lib.ntfp8_transpose(src.data_ptr(), rows, cols, store.data_ptr() + shift, nt.stream_ptr(dev)), "transpose")
        assert torch.equal(store[shift:shift + rows * cols].view(cols, rows), src.t())
        assert bool((store[:shift] == 7).all() and (store[shift + rows * cols:] == 7).all())


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_cast_with_transposed_copy(shape, dtype):
    from nanotron_amd.fp8 import DelayedScaling, DTypes, FP8Tensor

    x = (torch.randn(shape, generator=torch.Generator().manual_seed(shape[0])) * 3).to(dtype)
    x.view(-1)[-1] = 100.0   # the largest value in the last corner
    state = DelayedScaling(DTypes.FP8E4M3, 16, 0, "cuda")
    ref = O.DelayedScaling(O.E4M3)
    for step in range(2):    # current scaling first, then the fused delayed step
        print(f"cast {shape} {dtype} step {step}", flush=True)
        q = FP8Tensor(x.cuda(), DTypes.FP8E4M3, state=state, with_transpose=True)
        r = ref.quantise(x)
        assert state.initialised   # (the host knows of the scale: the next step is the fused one)
        assert torch.equal(q.cpu().as_subclass(torch.Tensor), r.q)
        assert torch.equal(q.transposed().cpu().as_subclass(torch.Tensor), r.q.t())
        assert q.fp8_meta.amax.item() == r.amax.item() and state.scale.item() == ref.scale.item()
