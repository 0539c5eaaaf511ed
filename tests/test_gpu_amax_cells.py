"""GPU parity of the maximum that the workgroups of a quantise launch put together: one word per workgroup up to 512 of them
(one, two, the last one short, exactly 512), which work through more tiles than that beyond; the largest element in the first, a middle and the last
workgroup; maxima that shrink from call to call, so that a word left behind by an earlier launch would show.  Exact."""
import pytest
import torch

from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu

FLAT = [(1, 7), (1, 32768), (1, 32769), (1, 98304), (2048, 4096)]   # 1, 1, 2, 3 and 256 workgroups of 32768 elements
# one element per thread; 64-wide tiles: 511, 512 and 520 of them; 128-wide ones: 512 and 768 (in 512 workgroups)
TILES = [(64, 64), (4672, 448), (4096, 512), (4160, 512), (4096, 2048), (4096, 3072)]


@pytest.mark.parametrize("shape,with_t", [(s, False) for s in FLAT] + [(s, True) for s in TILES])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_maximum_over_workgroups(shape, with_t, dtype):
    from nanotron_amd.fp8 import DelayedScaling, DTypes, FP8Tensor

    n = shape[0] * shape[1]
    base = torch.randn(shape, generator=torch.Generator().manual_seed(n)).clamp_(-3, 3).to(dtype)
    state, ref = DelayedScaling(DTypes.FP8E4M3, 2, 0, "cuda"), O.DelayedScaling(O.E4M3, 2)
    for peak, at in ((4096.0, 0), (1024.0, n - 1), (float("inf"), n // 2), (256.0, n // 2), (64.0, n - 1), (16.0, 0), (0.0, 0)):
        x = base.clone() if peak else torch.zeros_like(base)
        x.view(-1)[at] = peak
        print(f"{shape} {dtype} {peak} at {at}", flush=True)
        q, r = FP8Tensor(x.cuda(), DTypes.FP8E4M3, state=state, with_transpose=with_t), ref.quantise(x)
        assert q.fp8_meta.amax.item() == r.amax.item() == peak
        assert state.scale.item() == ref.scale.item()
        assert torch.equal(q.cpu().as_subclass(torch.Tensor), r.q)
        if with_t:
            assert torch.equal(q.transposed().cpu().as_subclass(torch.Tensor), r.q.t())
        assert state.initialised   # (asked once: the steps from here on take the fused entry point)
