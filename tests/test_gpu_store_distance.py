"""16-bit outputs are stored sixteen bytes a lane while the next block's values are computed in the same registers: what is
stored is the block's own, in every run.  Operands are small integers, so every sum is exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mnk", [(1712, 1056, 272), (1000, 1056, 512), (2064, 2080, 768), (1124, 5136, 512), (4100, 6160, 512), (64, 40, 77)])
@pytest.mark.parametrize("odt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bias", [True, False])
def test_every_run_stores_the_same_bits(mnk, odt, bias):
    from nanotron_amd import _native as nt

    M, N, K = mnk
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + N)
    a, b = (torch.randint(-3, 4, (r, K), generator=g, device=dev).float() for r in (M, N))
    bv = torch.randint(-4, 5, (N,), generator=g, device=dev).float() if bias else None
    want = ((a @ b.t()) + (bv if bias else 0)).to(odt)
    qa, qb = (t.to(torch.float8_e4m3fn).view(torch.uint8) for t in (a, b))
    one = torch.ones(1, device=dev)
    print(f"{mnk} {odt} bias={bias}", flush=True)
    bad = torch.zeros((), dtype=torch.int64, device=dev)
    for _ in range(40):
        bad += (nt.host.gemm(qa, nt.E4M3, one, qb, nt.E4M3, one, nt.TORCH_TO_NT[odt], None, False, bv, False) != want).sum()
    assert int(bad) == 0
