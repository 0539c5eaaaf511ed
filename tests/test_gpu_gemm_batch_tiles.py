"""Several problems in one launch, whatever tile size is chosen for them together: the results of the same problems one by one, bit
for bit.  Depths far apart (a few deep tiles beside many shallow ones), one to four problems, ragged edges."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BACKWARD = [(1024, 2048, 4864), (512, 1280, 4096), (768, 2048, 6912), (3856, 1856, 832), (336, 816, 3936), (2048, 1024, 1024), (272, 144, 4096),
            (2912, 2544, 3520), (1040, 3664, 3920), (3152, 2464, 3712)]   # ... with a few 256-wide tiles behind a round of them


def _operand(g, rows, cols):
    return (torch.randn(rows, cols, generator=g, device="cuda") * 8).to(torch.float8_e4m3fn).view(torch.uint8)


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("T,K,N", BACKWARD)
def test_backward_pair(T, K, N, accumulate):
    from nanotron_amd import _native as nt

    g = torch.Generator(device="cuda").manual_seed(T + N)
    one = torch.full((1,), 0.5, device="cuda")
    dy, w, x = _operand(g, T, N), _operand(g, N, K), _operand(g, T, K)
    base = torch.randn(N, K, generator=g, device="cuda") if accumulate else None
    print(f"{T} {K} {N} {accumulate}", flush=True)

    def problems():
        acc = base.clone() if accumulate else None
        return [(dy, 0, one, w, 0, one, nt.BF16, None, True, None, False), (dy, 0, one, x, 0, one, nt.F32, acc, True, None, True)]

    pair = nt.host.gemm_batch(problems())
    for got, p in zip(pair, problems()):
        assert torch.equal(got, nt.host.gemm(*p))


@pytest.mark.parametrize("count", [1, 2, 3, 4, 5])
def test_a_list_of_problems(count):
    from nanotron_amd import _native as nt

    g = torch.Generator(device="cuda").manual_seed(count)
    one = torch.full((1,), 0.5, device="cuda")
    shapes = [(300, 272, 2048), (1000, 528, 256), (2048, 1024, 640), (130, 4096, 384), (260, 1040, 1040)][:count]
    probs = [(_operand(g, M, K), 0, one, _operand(g, N, K), 0, one, (nt.F32, nt.BF16, nt.F16)[i % 3], None, False, None, False)
             for i, (M, N, K) in enumerate(shapes)]
    print(count, flush=True)
    for got, p in zip(nt.host.gemm_batch(probs), probs):
        assert torch.equal(got, nt.host.gemm(*p))
