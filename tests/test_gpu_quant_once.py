"""GPU parity of current scaling in one launch (small tensors), up to and just beyond the largest tensor it takes, with and
without the transposed copy, and of the cast that records its scale: exact."""
import pytest
import torch

from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (1, 17), (4, 16), (16, 16), (128, 128), (4096, 16), (4, 16384), (12, 5456), (255, 257), (256, 256), (256, 260), (1024, 65)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_current_scaling_and_first_use(shape, dtype):
    from nanotron_amd.fp8 import DelayedScaling, DTypes, FP8Tensor
    from nanotron_amd.fp8.tensor import cast_with_scale

    x = torch.randn(shape, generator=torch.Generator().manual_seed(shape[1])).to(dtype)
    bad = x.clone()
    bad.view(-1)[-1] = float("nan")
    for fmt, ofmt in ((DTypes.FP8E4M3, O.E4M3), (DTypes.FP8E5M2, O.E5M2)):
        for t in (x, bad, torch.zeros_like(x)):
            print(f"{shape} {dtype} {fmt}", flush=True)
            r = O.quantise_current(t, ofmt)
            for with_t in (False, True):
                q = FP8Tensor(t.cuda(), fmt, with_transpose=with_t)
                assert torch.equal(q.cpu().as_subclass(torch.Tensor), r.q)
                assert q.fp8_meta.scale.item() == r.scale.item()
                assert q.fp8_meta.amax.item() == r.amax.item() or t is bad and q.fp8_meta.amax.isnan()
                if with_t:
                    assert torch.equal(q.transposed().cpu().as_subclass(torch.Tensor), r.q.t())
        state, ref = DelayedScaling(fmt, 4, 0, "cuda"), O.DelayedScaling(ofmt, 4)
        for t in (torch.zeros_like(x), x, x * 3):
            # (the host does not ask for the flag here: every step takes the first-use entry point)
            q, r = FP8Tensor(t.cuda(), fmt, state=state), ref.quantise(t)
            assert torch.equal(q.cpu().as_subclass(torch.Tensor), r.q) and state.scale.item() == ref.scale.item()
            state._known = False
        c = cast_with_scale(x.cuda(), state.scale, fmt, with_transpose=True)
        assert torch.equal(c.cpu().as_subclass(torch.Tensor), O.cast_to_fp8(x, ref.scale, ofmt))
        assert torch.equal(c.transposed().cpu().as_subclass(torch.Tensor), O.cast_to_fp8(x, ref.scale, ofmt).t())
        assert c.fp8_meta.scale.item() == state.scale.item() and c.fp8_meta.amax.item() == 0.0
