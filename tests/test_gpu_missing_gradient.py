"""A consumer whose backward produces no gradient leaves the layer with a gradient of zeros, as autograd's own layers get."""
import pytest
import torch

pytestmark = pytest.mark.gpu


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.parametrize("delayed", [False, True])
def test_missing_gradient_counts_as_zeros(delayed):
    from nanotron_amd.fp8 import FP8Linear

    lin = FP8Linear(64, 96, True, torch.device("cuda", 0), delayed_scaling=delayed)
    x = torch.randn(32, 64, device="cuda", requires_grad=True)
    _NoGradient.apply(lin(x)).sum().backward()
    for g, like in ((x.grad, x), (lin.weight.grad, lin.weight), (lin.bias.grad, lin.bias)):
        assert g is not None and g.shape == like.shape and not bool(g.any())
