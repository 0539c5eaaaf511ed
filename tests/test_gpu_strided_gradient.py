"""Output gradients that do not lie contiguous (expanded by sum(), transposed views): the backward of a biased layer makes
one contiguous copy for the bias gradient and the quantisation together, and the results are those of the copy."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["expanded", "transposed", "3-D slice"])
def test_one_copy_of_a_strided_gradient(form):
    from nanotron_amd.fp8 import FP8Linear

    torch.manual_seed(7)
    lin = FP8Linear(96, 160, bias=True, device="cuda")
    if form == "3-D slice":
        x = torch.randn(5, 16, 96, device="cuda", requires_grad=True)
        g = torch.randn(5, 32, 160, device="cuda")[:, ::2]
    else:
        x = torch.randn(80, 96, device="cuda", requires_grad=True)
        g = torch.randn(160, 80, device="cuda").t() if form == "transposed" else torch.full((1, 1), 0.5, device="cuda").expand(80, 160)
    assert not g.is_contiguous()

    def step(grad):
        lin.weight.grad = lin.bias.grad = x.grad = None
        y = lin(x)
        torch.cuda.synchronize()
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        y.backward(grad)
        made = torch.cuda.memory_stats()["allocation.all.allocated"] - before
        return made, [x.grad.clone(), lin.weight.grad.clone(), lin.bias.grad.clone()]

    dense = g.contiguous()
    step(dense)
    plain, want = step(dense)
    strided, got = step(g)
    assert strided == plain + 1
    for a, b in zip(got, want):
        assert torch.equal(a, b)
