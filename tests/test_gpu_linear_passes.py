"""A layer's passes through one native call each against the same passes put together from their pieces: outputs, gradients,
fp8 bytes and scaling states bit for bit, over the forms that the operands take (read as they are, transposed copies, any
sizes), and the calls that must not take the short way."""
import pytest
import torch
from torch.autograd import forward_ad

from nanotron_amd.fp8 import DTypes, FP8Linear, FP8Parameter
from nanotron_amd.fp8 import linear as L


class _Spy:
    """Which calls of the native forward and backward were served, in order, and which of the latter were to send an fp8 dX."""

    def __init__(self, monkeypatch):
        self.forward, self.backward, self.fp8 = [], [], []
        fwd, bwd = L._quantise_and_multiply, L._backward_passes

        def forward(*a):
            res = fwd(*a)
            self.forward.append(res is not None)
            return res

        def backward(*a):
            res = bwd(*a)
            self.backward.append(res is not None)
            self.fp8.append(a[-1] is not None)
            return res

        monkeypatch.setattr(L, "_quantise_and_multiply", forward)
        monkeypatch.setattr(L, "_backward_passes", backward)


def _run(x, gys, dtype, out, bias, delayed, accumulate, dims, pieces, monkeypatch, offset=0):
    if pieces:
        monkeypatch.setattr(L, "_quantise_and_multiply", lambda *a: None)
        monkeypatch.setattr(L, "_backward_passes", lambda *a: None)
    spy = _Spy(monkeypatch)
    K, N = x.shape[-1], gys[0].shape[-1]
    g = torch.Generator(device="cuda").manual_seed(3)
    lin = FP8Linear(K, N, bias, "cuda", dtype=dtype, out_dtype=out, delayed_scaling=delayed, accumulate_grad=accumulate)
    lin.weight = FP8Parameter((torch.randn(N, K, generator=g, device="cuda") * 0.02).to(dtype), DTypes.FP8E4M3)
    if bias:
        lin.bias.data.copy_(torch.randn(N, generator=g, device="cuda") * 0.02)
    got = []
    for gy in gys:
        xg = torch.empty(x.numel() + offset, dtype=dtype, device="cuda")[offset:].view(x.shape).copy_(x).requires_grad_(True)
        y = lin(xg)
        saved = y.grad_fn.saved_tensors[0]
        got += [y.detach().clone(), saved.as_subclass(torch.Tensor).clone(), saved.fp8_meta.scale.clone()]
        y.backward(gy)
        torch.cuda.synchronize()
        got += [xg.grad, (lin.weight.grad if dtype == torch.float32 else lin.weight.main_grad).clone()]
        if bias:
            got.append(lin.bias.grad.clone())
            lin.bias.grad = None
        if delayed:
            got += [r._buf.clone() for r in lin.scaling.values()]
    lin.eval()
    with torch.no_grad():
        got.append(lin(x))
    got.append(lin(x).detach())
    if delayed:
        got += [r._buf.clone() for r in lin.scaling.values()]
    monkeypatch.undo()
    # the first use of a scaling role takes the pieces, every other pass is served; without gradients a pass that is not
    # served asks once more inside autograd's function
    steps = [not pieces and (i > 0 or not delayed) for i in range(len(gys))]
    assert spy.backward == steps and spy.forward == steps + ([False] * 3 if pieces else [True] * 2)
    return got


CASES = [
    # tokens, K, N, dtype, out, bias, delayed, accumulate, dims
    (128, 128, 128, torch.float32, None, True, False, False, 2),
    (256, 144, 272, torch.bfloat16, torch.bfloat16, True, True, True, 2),
    (512, 256, 384, torch.bfloat16, torch.float32, False, True, True, 3),
    (1021, 256, 320, torch.float16, torch.float16, True, True, False, 2),
    (77, 130, 91, torch.float32, torch.float32, True, True, True, 3),
    (96, 515, 601, torch.float16, torch.float16, False, False, True, 2),
    (1, 64, 48, torch.bfloat16, torch.bfloat16, True, False, False, 1),
    (300, 256, 264, torch.bfloat16, torch.bfloat16, False, True, False, 2),
]


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("tokens,K,N,dtype,out,bias,delayed,accumulate,dims", CASES)
def test_same_as_the_pieces(tokens, K, N, dtype, out, bias, delayed, accumulate, dims, offset, monkeypatch):
    g = torch.Generator(device="cuda").manual_seed(tokens)
    lead = {1: (), 2: (tokens,), 3: (1, tokens)}[dims]
    x = torch.randn(*lead, K, generator=g, device="cuda").to(dtype)
    gys = [(torch.randn(*lead, N, generator=g, device="cuda") * 1e-3).to(out or torch.float32) for _ in range(4)]
    if tokens == 300:   # a strided gradient
        gys = [torch.stack([t, t], -1)[..., 0] for t in gys]
    args = (x, gys, dtype, out, bias, delayed, accumulate, dims)
    short = _run(*args, False, monkeypatch, offset)
    pieces = _run(*args, True, monkeypatch, offset)
    assert len(short) == len(pieces)
    for i, (a, b) in enumerate(zip(short, pieces)):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), i


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,K,N", [(1, 1024, 1024), (16, 1024, 1024), (100, 1024, 1024), (128, 1024, 2304), (112, 144, 256), (129, 144, 256)])
@pytest.mark.parametrize("bias", [False, True])
def test_few_tokens(tokens, K, N, bias, monkeypatch):
    """A weight that more than 128 tokens read as it is: its transposed copy, gone with every re-quantisation, is made inside
    the native pass."""
    res = []
    for pieces in (False, True):
        g = torch.Generator(device="cuda").manual_seed(tokens)
        torch.manual_seed(3)   # (the bias)
        lin = FP8Linear(K, N, bias, "cuda", dtype=torch.bfloat16, out_dtype=torch.bfloat16, delayed_scaling=True)
        lin.weight = FP8Parameter((torch.randn(N, K, generator=g, device="cuda") * 0.02).to(torch.bfloat16), DTypes.FP8E4M3)
        assert getattr(lin.weight.data, "_transposed", None) is None
        got = []
        for step in range(3):
            if pieces:
                monkeypatch.setattr(L, "_quantise_and_multiply", lambda *a: None)
                monkeypatch.setattr(L, "_backward_passes", lambda *a: None)
            spy = _Spy(monkeypatch)
            lin.requantize_weight()
            assert getattr(lin.weight.data, "_transposed", None) is None
            x = torch.randn(tokens, K, generator=g, device="cuda").to(torch.bfloat16).requires_grad_(True)
            y = lin(x)
            y.backward((torch.randn(tokens, N, generator=g, device="cuda") * 1e-3).to(torch.bfloat16))
            torch.cuda.synchronize()
            monkeypatch.undo()
            assert spy.backward == [step > 0 and not pieces]
            assert (getattr(lin.weight.data, "_transposed", None) is not None) == (tokens <= 128)
            if tokens <= 128:
                got.append(lin.weight.data._transposed.as_subclass(torch.Tensor))
                assert torch.equal(got[-1], lin.weight.data.as_subclass(torch.Tensor).t())
                assert lin.weight.data._transposed.fp8_meta is lin.weight.data.fp8_meta
            got += [y.detach(), x.grad, lin.weight.main_grad] + [r._buf.clone() for r in lin.scaling.values()]
        res.append(got)
    for i, (a, b) in enumerate(zip(*res)):
        assert torch.equal(a, b), i


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,bias", [(258, False), (301, False), (100, False), (77, False), (256, True), (301, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_ragged_chain_is_served(tokens, bias, dtype, monkeypatch):
    """An fp8 gradient of a token count that is no multiple of 4 or 16: copies of the weight, of the fp8 input and of the fp8
    gradient are made inside the native passes; a bias gradient summed from fp8 values.  With the results of the pieces."""
    res = []
    for pieces in (False, True):
        g = torch.Generator(device="cuda").manual_seed(tokens)
        torch.manual_seed(3)   # (the biases)
        lins = [FP8Linear(a, b, bias, "cuda", dtype=dtype, out_dtype=o, delayed_scaling=True)
                for a, b, o in ((256, 384, DTypes.FP8E4M3), (384, 272, torch.bfloat16))]
        for lin in lins:
            lin.weight = FP8Parameter((torch.randn(lin.weight.shape, generator=g, device="cuda") * 0.05).to(dtype), DTypes.FP8E4M3)
        got = []
        for step in range(3):
            if pieces:
                monkeypatch.setattr(L, "_quantise_and_multiply", lambda *a: None)
                monkeypatch.setattr(L, "_backward_passes", lambda *a: None)
            spy = _Spy(monkeypatch)
            for lin in lins:
                lin.requantize_weight()
            x = torch.randn(tokens, 256, generator=g, device="cuda").to(torch.bfloat16).requires_grad_(True)
            y = lins[1](lins[0](x))
            y.backward((torch.randn(tokens, 272, generator=g, device="cuda") * 1e-3).to(torch.bfloat16))
            torch.cuda.synchronize()
            monkeypatch.undo()
            assert spy.fp8 == [step > 0, False] and spy.backward == [step > 0 and not pieces] * 2
            got += [y.detach(), x.grad] + [lin.weight.grad if dtype == torch.float32 else lin.weight.main_grad for lin in lins] + [r._buf.clone() for lin in lins for r in lin.scaling.values()]
            if bias:
                got += [lin.bias.grad.clone() for lin in lins]
        res.append(got)
    for i, (a, b) in enumerate(zip(*res)):
        assert torch.equal(a, b), i


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,dims,delayed", [(512, (256, 384), True), (300, (256, 384), False), (77, (130, 91), True), (258, (256, 384, 272), True), (256, (256, 384, 272), True)])
def test_quantised_gradient_kept_on_request(tokens, dims, delayed, monkeypatch):
    """The e5m2 output gradient that a checker asks for is the one that the native passes multiply."""
    res = []
    for pieces in (False, True):
        g = torch.Generator(device="cuda").manual_seed(tokens)
        lins = []
        for i, (a, b) in enumerate(zip(dims, dims[1:])):
            out = torch.bfloat16 if i == len(dims) - 2 else DTypes.FP8E4M3
            lin = FP8Linear(a, b, False, "cuda", dtype=torch.bfloat16, out_dtype=out, delayed_scaling=delayed)
            lin.weight = FP8Parameter((torch.randn(b, a, generator=g, device="cuda") * 0.05).to(torch.bfloat16), DTypes.FP8E4M3)
            lin.keep_quantised_grad = True
            lins.append(lin)
        got = []
        for step in range(2):
            if pieces:
                monkeypatch.setattr(L, "_backward_passes", lambda *a: None)
            spy = _Spy(monkeypatch)
            h = torch.randn(tokens, dims[0], generator=g, device="cuda").to(torch.bfloat16).requires_grad_(True)
            for lin in lins:
                h = lin(h)
            h.backward((torch.randn(tokens, dims[-1], generator=g, device="cuda") * 1e-3).to(torch.bfloat16))
            torch.cuda.synchronize()
            monkeypatch.undo()
            assert spy.backward == [not pieces and (step > 0 or not delayed)] * len(lins)
            for lin in lins:
                q, lin.quantised_grad_output = lin.quantised_grad_output, None
                assert q.fp8_meta.dtype is DTypes.FP8E5M2 and q.shape == (tokens, lin.weight.shape[0])
                t = getattr(q, "_transposed", None)
                got += [q.as_subclass(torch.Tensor), q.fp8_meta.amax, q.fp8_meta.scale, torch.tensor(t is not None)]
                if t is not None:
                    got.append(t.as_subclass(torch.Tensor))
                    assert torch.equal(got[-1], got[-5].t())
        res.append(got)
    assert len(res[0]) == len(res[1])
    for i, (a, b) in enumerate(zip(*res)):
        assert a.shape == b.shape and torch.equal(a, b), i


@pytest.mark.gpu
def test_frozen_weight_and_input_without_gradient(monkeypatch):
    x = torch.randn(256, 256, device="cuda", dtype=torch.bfloat16)
    gy = torch.randn(256, 384, device="cuda", dtype=torch.bfloat16)
    for frozen in (False, True):
        res = []
        for pieces in (False, True):
            if pieces:
                monkeypatch.setattr(L, "_backward_passes", lambda *a: None)
            torch.manual_seed(0)
            lin = FP8Linear(256, 384, True, "cuda", dtype=torch.bfloat16, out_dtype=torch.bfloat16)
            lin.weight.requires_grad_(not frozen)
            xg = x.clone().requires_grad_(frozen)
            spy = _Spy(monkeypatch)
            lin(xg).backward(gy)
            assert spy.forward == [True] and spy.backward == [not pieces]
            assert (xg.grad is None) == (not frozen) and (getattr(lin.weight, "main_grad", None) is None) == frozen
            res.append([xg.grad if frozen else lin.weight.main_grad, lin.bias.grad])
            monkeypatch.undo()
        assert all(torch.equal(a, b) for a, b in zip(*res))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,dims,bias", [(512, (256, 384, 272), False), (300, (256, 320, 272), False), (258, (272, 320, 256), True), (64, (128, 96, 112), False)])
def test_chain_same_as_the_pieces(tokens, dims, bias, monkeypatch):
    """fp8 activations forward and e5m2 gradients back, at sizes that are read as they are and others."""
    res = []
    for pieces in (False, True):
        if pieces:
            monkeypatch.setattr(L, "_quantise_and_multiply", lambda *a: None)
            monkeypatch.setattr(L, "_backward_passes", lambda *a: None)
        spy = _Spy(monkeypatch)
        g = torch.Generator(device="cuda").manual_seed(tokens)
        lins = []
        for i, (a, b) in enumerate(zip(dims, dims[1:])):
            lin = FP8Linear(a, b, bias, "cuda", dtype=torch.bfloat16, out_dtype=DTypes.FP8E4M3 if i == 0 else torch.bfloat16, delayed_scaling=True)
            lin.weight = FP8Parameter((torch.randn(b, a, generator=g, device="cuda") * 0.05).to(torch.bfloat16), DTypes.FP8E4M3)
            if bias:
                lin.bias.data.zero_()
            lins.append(lin)
        got = []
        for step in range(3):
            x = torch.randn(tokens, dims[0], generator=g, device="cuda").to(torch.bfloat16).requires_grad_(True)
            h = x
            for lin in lins:
                h = lin(h)
            h.backward((torch.randn(tokens, dims[-1], generator=g, device="cuda") * 1e-3).to(torch.bfloat16))
            torch.cuda.synchronize()
            got += [h.detach(), x.grad] + [lin.weight.main_grad for lin in lins] + [r._buf.clone() for lin in lins for r in lin.scaling.values()]
            if bias:
                got += [lin.bias.grad.clone() for lin in lins]
        got.append(torch.tensor([lin.fp8_grad_inputs_sent for lin in lins]))
        res.append(got)
        monkeypatch.undo()
        # the last layer first; an fp8 output is not the native forward's, nor is the pass over an fp8 input
        assert spy.fp8 == [False, False, True, False, True, False] and spy.forward == [False] * 3
        assert spy.backward == [False] * 2 + [not pieces] * 4
    for i, (a, b) in enumerate(zip(*res)):
        assert torch.equal(a, b), i


@pytest.mark.gpu
def test_evaluation_with_a_scale_held_on_another_device():
    """A layer whose scaling roles were kept on the host after training evaluates with the scale they hold."""
    lin = FP8Linear(256, 384, False, "cuda", dtype=torch.bfloat16, out_dtype=torch.bfloat16, delayed_scaling=True)
    x = torch.randn(64, 256, device="cuda", dtype=torch.bfloat16)
    lin(x)
    torch.cuda.synchronize()
    lin.eval()
    with torch.no_grad():
        want = lin(x)
        state = lin.scaling["input"]
        assert state.known_initialised
        state._buf = state._buf.cpu()
        assert torch.equal(lin(x), want)
    assert torch.equal(lin(x).detach(), want)


@pytest.mark.gpu
def test_saved_tensor_hooks_see_what_a_layer_saves():
    lin = FP8Linear(256, 256, False, "cuda", out_dtype=torch.float32)
    x = torch.randn(256, 256, device="cuda", requires_grad=True)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
        y = lin(x)
    assert any(t.dtype == torch.uint8 and t.shape == x.shape for t in packed)
    with pytest.raises(AssertionError, match="FP8Tensors"):   # hooks hand back the weight's storage, not the parameter
        y.sum().backward()


def test_transforms_are_seen():
    assert L._no_transform()
    with forward_ad.dual_level():
        assert not L._no_transform()
    seen = []
    torch.func.vmap(lambda t: seen.append(L._no_transform()) or t)(torch.zeros(2))
    torch.jit.trace(lambda t: seen.append(L._no_transform()) or t + 1, torch.zeros(2), check_trace=False)
    assert seen == [False, False] and L._no_transform()


@pytest.mark.parametrize("owner,name", [(forward_ad, "_current_level"), (torch._C._functorch, "peek_interpreter_stack"), (torch._C, "_get_tracing_state"),
                                        (torch._C, "_functorch")])
def test_a_torch_that_does_not_tell_of_transforms(owner, name, monkeypatch):
    """Without one of the private names the way past autograd is not taken; nothing raises."""
    import importlib.util

    spec = importlib.util.spec_from_file_location("linear_elsewhere", L.__file__)
    module = importlib.util.module_from_spec(spec)
    monkeypatch.delattr(owner, name)
    spec.loader.exec_module(module)
    assert not module._no_transform()
    monkeypatch.undo()
    assert L._no_transform()


@pytest.mark.gpu
def test_gemm_observer_sees_the_calls_of_the_native_passes(monkeypatch):
    from nanotron_amd import _native as nt

    T, K, N = 256, 384, 272
    x = torch.randn(T, K, device="cuda", dtype=torch.bfloat16)
    gy = torch.randn(T, N, device="cuda", dtype=torch.bfloat16)
    res, seen = [], []
    for watch in (False, True):
        torch.manual_seed(0)
        lin = FP8Linear(K, N, False, "cuda", dtype=torch.bfloat16, out_dtype=torch.bfloat16)
        spy = _Spy(monkeypatch)
        assert nt.host.set_gemm_observer((lambda *a: seen.append(a)) if watch else None) is None
        xg = x.clone().requires_grad_(True)
        y = lin(xg)
        y.backward(gy)
        assert (nt.host.set_gemm_observer(None) is not None) == watch
        monkeypatch.undo()
        assert spy.forward == [True] and spy.backward == [True]
        res.append([y.detach(), xg.grad, lin.weight.main_grad])
    forward, backward = ((T, N, K),), ((T, K, N), (N, K, T))
    assert seen == [(False, forward), (True, forward), (False, backward), (True, backward)]
    assert all(torch.equal(a, b) for a, b in zip(*res))

    # whoever is told may drop the workspaces: an fp8 output's bookkeeping takes its own afterwards
    fp8 = []
    for watch in (False, True):
        torch.manual_seed(0)
        out = FP8Linear(K, N, False, "cuda", dtype=torch.bfloat16, out_dtype=DTypes.FP8E4M3, delayed_scaling=True)
        out(x)
        torch.cuda.synchronize()
        nt.host.set_gemm_observer((lambda *a: nt.host.drop_workspaces()) if watch else None)
        try:
            q = out(x)
        finally:
            nt.host.set_gemm_observer(None)
        fp8.append([q.as_subclass(torch.Tensor), q.fp8_meta.amax, out.scaling["output"]._buf])
        assert float(q.fp8_meta.amax) > 0
    assert all(torch.equal(a, b) for a, b in zip(*fp8))

    def refuse(*a):
        raise ValueError("no")

    nt.host.set_gemm_observer(refuse)
    try:
        with pytest.raises(ValueError, match="no"):
            lin(x)
    finally:
        nt.host.set_gemm_observer(None)
    with torch.no_grad():
        assert torch.equal(lin(x), res[0][0])
    with pytest.raises(TypeError):
        nt.host.set_gemm_observer(3)
