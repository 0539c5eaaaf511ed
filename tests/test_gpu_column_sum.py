"""GPU parity of the column sums (the bias gradient) at the edges of their 64-column blocks and row runs, against an fp64
sum: fp32 sums of `rows` terms lie within rows * 2^-24 * sum|x| of it, plus one rounding to the output type.  Two runs
give the same bits (the order of the sum depends on the shape alone)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (15, 64), (17, 65), (64, 63), (65, 4), (128, 128), (1021, 2304), (4096, 130), (777, 33000), (100000, 7)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_sums(shape, dtype):
    from nanotron_amd import _native as nt

    x = torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(shape[0]), device="cuda").to(dtype)
    ref, mag = x.double().sum(0), x.double().abs().sum(0)
    for odt, step in ((torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -10)):
        print(f"{shape} {dtype} -> {odt}", flush=True)
        got = nt.host.column_sum(x, nt.TORCH_TO_NT[odt])
        assert got.dtype == odt and got.shape == (shape[1],)
        slack = shape[0] * 2.0 ** -24 * mag
        assert bool(((got.double() - ref).abs() <= slack + step * (ref.abs() + slack) + 2.0 ** -24).all())
        assert torch.equal(got, nt.host.column_sum(x, nt.TORCH_TO_NT[odt]))
