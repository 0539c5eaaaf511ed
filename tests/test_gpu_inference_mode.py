"""Validation under torch.inference_mode() before training: nothing that a layer keeps from it may stop it from training."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _chain():
    from nanotron_amd.fp8 import DTypes, FP8Linear

    torch.manual_seed(5)
    return [FP8Linear(64, 128, bias=True, device="cuda", out_dtype=DTypes.FP8E4M3, delayed_scaling=True, amax_history_len=4),
            FP8Linear(128, 64, bias=False, device="cuda", delayed_scaling=True, amax_history_len=4)]


def _step(chain, x):
    x.grad = None
    y = chain[1](chain[0](x))
    y.backward(torch.ones_like(y))
    return [y.detach(), x.grad.clone(), chain[0].weight.grad.clone(), chain[1].weight.grad.clone(), chain[0].bias.grad.clone()]


@pytest.mark.parametrize("eval_mode", [True, False])
def test_inference_mode_first_then_training(eval_mode):
    x = torch.randn(48, 64, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    chain, twin = _chain(), _chain()
    for mods, mode in ((chain, torch.inference_mode), (twin, torch.no_grad)):
        for m in mods:
            m.train(not eval_mode)
        with mode():
            mods[1](mods[0](x))
        for m in mods:
            m.train()
    xa, xb = (x.clone().requires_grad_(True) for _ in range(2))
    for step in range(3):   # (from the second step on the second layer's gradient goes back in fp8)
        for m in chain + twin:
            m.weight.grad = None
            if m.bias is not None:
                m.bias.grad = None
        for a, b in zip(_step(chain, xa), _step(twin, xb)):
            assert torch.equal(a, b), step
        for m in chain + twin:
            assert m.scaling["output_grad"].initialised   # (asked: the next step sends gradients in fp8)
    assert chain[1].fp8_grad_inputs_sent == twin[1].fp8_grad_inputs_sent > 0


def test_gradient_handle_after_inference_mode_is_part_of_the_graph():
    """The handle of an fp8 output may be reshaped on its way to the next layer: that is an operation autograd records."""
    lin, twin = _chain()[0], _chain()[0]
    x = torch.randn(48, 64, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    with torch.inference_mode():
        lin(x)
    with torch.no_grad():
        twin(x)
    for m in (lin, twin):
        handle = m(x)._grad_handle
        assert not handle.is_inference()
        handle.reshape(6, 8, 128).mul(2.0).sum().backward()
    assert torch.equal(lin.weight.grad, twin.weight.grad) and torch.equal(lin.bias.grad, twin.bias.grad)
    assert float(lin.bias.grad[0]) == 96.0
