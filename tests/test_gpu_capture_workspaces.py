"""Graphs captured without a warm-up on their capture stream: each brings the zeroed workspaces it needs, whichever is
replayed first, and leaves those of eager calls on the same stream alone."""
import pytest
import torch

from nanotron_amd import _native as nt

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _dirty(pool, stream):
    """Leave words that look like arrived maxima in the small blocks of a graph memory pool."""
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, pool=pool, stream=stream):
        blocks = [torch.full((1 << 16,), -1, dtype=torch.int32, device=DEV) for _ in range(7)]
    g.replay()
    torch.cuda.synchronize()
    del blocks
    return g


@pytest.mark.parametrize("batch", [False, True])
def test_two_captures_the_second_replayed_first(batch):
    from nanotron_amd.fp8 import DelayedScaling, DTypes, FP8Tensor
    from nanotron_amd.fp8.tensor import quantize_delayed_batch

    x = torch.randn(512, 512, device=DEV).clamp_(-3, 3)
    x[17, 5] = 5.0

    def quantise(states):
        if batch:
            return quantize_delayed_batch([x] * 3, DTypes.FP8E4M3, states, [False] * 3)
        return [FP8Tensor(x, DTypes.FP8E4M3, state=states[0], with_transpose=True)]

    def roles():
        made = [DelayedScaling(DTypes.FP8E4M3, 4, 0, DEV) for _ in range(3)]
        for s in made:
            FP8Tensor(x, DTypes.FP8E4M3, state=s)
            assert s.initialised
        return made

    stream, pool = torch.cuda.Stream(), torch.cuda.graph_pool_handle()
    dirty = _dirty(pool, stream)
    graphs, outs, states = [], [], []
    for _ in range(2):
        states.append(roles())
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, pool=pool, stream=stream):
            outs.append(quantise(states[-1]))
        graphs.append(g)
    want = quantise(roles())
    eager = roles()
    for which in (1, 0, 1, 1, 0):
        graphs[which].replay()
        torch.cuda.synchronize()
        for q, w, s in zip(outs[which], want, states[which]):
            assert q.fp8_meta.amax.item() == 5.0
            assert torch.equal(q.as_subclass(torch.Tensor), w.as_subclass(torch.Tensor))
            assert s.amax_history[0].item() == 5.0
        with torch.cuda.stream(stream):   # eager work on the capture stream in between
            for q in quantise(eager):
                assert q.fp8_meta.amax.item() == 5.0
            assert int(nt.workspace_and_stream(DEV)[0].abs().sum()) == 0
            assert int(nt.workspace_pool(DEV, 3)[0].abs().sum()) == 0
        torch.cuda.synchronize()
    del dirty
