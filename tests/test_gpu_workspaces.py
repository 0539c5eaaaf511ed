"""The reduction workspaces that Python hands out are the ones that the native host calls use, and every kind of launch
leaves them zero: words of quantise launches, tickets of column sums, maxima and tickets of fp8-output GEMMs."""
import pytest
import torch

from nanotron_amd import _native as nt

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _allocations():
    return torch.cuda.memory_stats()["allocation.all.allocated"]


def test_one_table_of_workspaces():
    from nanotron_amd.fp8 import DelayedScaling, DTypes, FP8Tensor
    from nanotron_amd.fp8.kernel import fp8_matmul_kernel
    from nanotron_amd.fp8.tensor import quantize_delayed_batch

    s = torch.cuda.Stream()
    xs = [torch.randn(512, 512, device=DEV, dtype=torch.bfloat16) * (i + 1) for i in range(20)]
    states = [DelayedScaling(DTypes.FP8E4M3, 4, 0, DEV) for _ in xs]
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for x, st in zip(xs, states):
            FP8Tensor(x, DTypes.FP8E4M3, state=st)
            assert st.initialised
        before = _allocations()
        ws, stream = nt.workspace_and_stream(DEV)
        assert _allocations() == before, "the quantisations' own workspace, not another one"
        assert stream == s.cuda_stream

        quantize_delayed_batch(xs, DTypes.FP8E4M3, states, [False] * len(xs))
        before = _allocations()
        pool, _ = nt.workspace_pool(DEV, len(xs))
        assert _allocations() == before, "the batched call's own workspaces"
        assert pool.shape[0] >= len(xs) and int(pool.abs().sum()) == 0

        FP8Tensor(xs[0], DTypes.FP8E4M3, state=states[0])                                        # one word per workgroup
        assert int(ws.abs().sum()) == 0
        FP8Tensor(torch.randn(4096, 3072, device=DEV), DTypes.FP8E4M3, state=states[0], with_transpose=True)   # of two per CU
        assert int(ws.abs().sum()) == 0
        nt.host.column_sum(torch.randn(4096, 256, device=DEV), nt.F32)                           # tickets of the column blocks
        assert int(ws.abs().sum()) == 0
        q = FP8Tensor(xs[1], DTypes.FP8E4M3)
        fp8_matmul_kernel(q, True, q, False, False, out_dtype=DTypes.FP8E4M3, out_state=states[1])   # maxima, tickets
        assert int(ws.abs().sum()) == 0
    assert nt.workspace_and_stream(DEV)[0].data_ptr() != ws.data_ptr()
    torch.cuda.current_stream().wait_stream(s)
