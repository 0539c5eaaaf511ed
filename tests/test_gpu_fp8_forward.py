"""Layers that take or hand on fp8 activations, forward through one native call, against the same passes put together from their
pieces: bytes, transposed copies, gradients and scaling states bit for bit; and the passes that have to take the pieces."""
import pytest
import torch

from nanotron_amd.fp8 import DTypes, FP8Linear, FP8Parameter
from nanotron_amd.fp8 import linear as L
from nanotron_amd.fp8.optim import requantize_fp8_weights

pytestmark = pytest.mark.gpu


def _chain(dims, outs, dtype, bias, transpose, delayed):
    g = torch.Generator(device="cuda").manual_seed(5)
    lins = []
    for a, b, out in zip(dims, dims[1:], outs):
        lin = FP8Linear(a, b, bias, "cuda", dtype=dtype, out_dtype=out, delayed_scaling=delayed, fp8_output_transpose=transpose)
        lin.weight = FP8Parameter((torch.randn(b, a, generator=g, device="cuda") * 0.05).to(dtype), DTypes.FP8E4M3)
        if bias:
            lin.bias.data.copy_(torch.randn(b, generator=g, device="cuda") * 0.1)
        lins.append(lin)
    return lins


def _run(shape, dims, outs, dtype, bias, transpose, delayed, steps, native, monkeypatch):
    served = []
    real = L._multiply_fp8

    def spy(*a):
        res = real(*a) if native else None
        served.append(res is not None)
        return res

    monkeypatch.setattr(L, "_multiply_fp8", spy)
    lins = _chain(dims, outs, dtype, bias, transpose, delayed)
    g = torch.Generator(device="cuda").manual_seed(7)
    got = []
    for _ in range(steps):
        requantize_fp8_weights(lins)
        x = torch.randn(*shape, dims[0], generator=g, device="cuda").to(dtype)
        if len(shape) == 1 and shape[0] == 300:   # rows apart from each other
            x = torch.cat([x, x], 1)[:, :dims[0]]
        x.requires_grad_(True)
        h = x
        for lin in lins:
            h = lin(h)
            if type(h) is not torch.Tensor:
                got += [h.as_subclass(torch.Tensor), h.fp8_meta.amax, h.fp8_meta.scale]
                t = getattr(h, "_transposed", None)
                assert (t is not None) == transpose
                if t is not None:
                    got.append(t.as_subclass(torch.Tensor))
        h.backward((torch.randn(h.shape, generator=g, device="cuda") * 1e-3).to(h.dtype))
        torch.cuda.synchronize()
        got += [h.detach(), x.grad]
        got += [(lin.weight.grad if dtype == torch.float32 else lin.weight.main_grad).clone() for lin in lins]
        got += [r._buf.clone() for lin in lins if delayed for r in lin.scaling.values()]
        for lin in lins:
            lin.weight.grad = None
    for lin in lins:
        lin.eval()
    h = x.detach()
    for lin in lins:
        h = lin(h)
    got.append(h.detach())
    monkeypatch.undo()
    return got, served


E4, E5, BF, F32 = DTypes.FP8E4M3, DTypes.FP8E5M2, torch.bfloat16, torch.float32


@pytest.mark.parametrize("shape,dims,outs,dtype,bias,transpose", [
    ((256,), (256, 384, 384, 272), (E4, E4, BF), BF, False, False),
    ((2, 128), (256, 272, 144), (E4, BF), BF, True, True),
    ((300,), (256, 384, 272), (E5, F32), F32, False, True),
    ((77,), (130, 96, 91), (E4, F32), F32, True, False),
    ((1,), (64, 48, 32), (E4, BF), BF, False, False),
])
def test_same_as_the_pieces(shape, dims, outs, dtype, bias, transpose, monkeypatch):
    args = (shape, dims, outs, dtype, bias, transpose, True, 3)
    short, served = _run(*args, True, monkeypatch)
    pieces, _ = _run(*args, False, monkeypatch)
    n = len(outs)
    # a role's first use takes the pieces, and so does an fp8 output of an evaluation pass
    assert served[n:3 * n] == [True] * (2 * n) and served[3 * n:] == [False] * (n - 1) + [True]
    assert served[:n] == [False] * (n - 1) + [True]
    assert len(short) == len(pieces)
    for i, (a, b) in enumerate(zip(short, pieces)):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), i


def test_without_held_scales_the_pieces_are_taken(monkeypatch):
    args = ((128,), (128, 128, 64), (E4, BF), BF, False, False, False, 2)
    short, served = _run(*args, True, monkeypatch)
    pieces, _ = _run(*args, False, monkeypatch)
    assert served == [False, True] * 3
    assert all(torch.equal(a, b) for a, b in zip(short, pieces))


def test_what_does_not_fit_is_refused_as_before():
    lin = _chain((128, 64), (BF,), BF, False, False, True)[0]
    from nanotron_amd.fp8 import FP8Tensor

    q = FP8Tensor(torch.randn(32, 96, device="cuda"), E4)
    with pytest.raises(AssertionError, match="fit together"):
        lin(q)
