"""GPU parity of the dequantisation kernel at the edges of its 16-byte groups and of its grid, for outputs and inputs
that start anywhere: bit for bit the oracle's number for every code (src/nanotron/fp8/tensor.py:68-74)."""
import pytest
import torch

from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("odt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fmt", [O.E4M3, O.E5M2])
def test_sizes_and_alignments(fmt, odt):
    from nanotron_amd import _native as nt

    dev = torch.device("cuda", 0)
    scale = torch.tensor([2.0 ** 3])
    cases = [(n, 0, 0) for n in (1, 3, 4, 7, 8, 9, 255, 2047, 2049, 8191, 8193, 2 ** 21, 2 ** 21 + 5, 2 ** 22, 2 ** 22 + 9, 256 * 32 * 8192 + 5)] + [(4099, 1, 0), (4099, 3, 1), (4099, 0, 2), (64, 5, 0)]
    for n, i_shift, o_shift in cases:
        codes = (torch.arange(n + i_shift) * 37 % 256).to(torch.uint8)
        q = codes.to(dev)[i_shift:]
        store = torch.full((n + o_shift + 8,), 7.0, dtype=odt, device=dev)
        out = store[o_shift:o_shift + n]
        print(f"n={n} fmt={fmt} {odt} shifts {i_shift} {o_shift}", flush=True)
        nt.check(nt.lib.ntfp8_cast_from_fp8(q.data_ptr(), 0 if fmt == O.E4M3 else 1, scale.to(dev).data_ptr(), n, out.data_ptr(),
                                            nt.TORCH_TO_NT[odt], nt.stream_ptr(dev)), "cast")
        table = O.cast_from_fp8(torch.arange(256).to(torch.uint8), scale[0], fmt, odt)
        want = table[codes[i_shift:].long()]
        bits = torch.int32 if odt == torch.float32 else torch.int16
        got = out.cpu().contiguous()
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        number = ~torch.isnan(want)   # (the payload of a NaN is the hardware's)
        assert torch.equal(got.view(bits)[number], want.view(bits)[number]), (n, i_shift, o_shift)
        assert bool((store[o_shift + n:] == 7).all() and (store[:o_shift] == 7).all())
