"""GPU parity of GEMMs whose K is not a multiple of 16 or whose pointers are not aligned (`gemm_any_kernel`), at the
edges of its tiles (64 or 128 wide, 128 bytes of K, 16-byte chunks).  Reference: an fp64 product of the exactly-upcast
operands.  The kernel's products are exact and its sum is rounded at most once per product and once per step, so every
element lies within K * 2^-23 * (|A| . |B|^T) of the reference."""
import pytest
import torch

from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu


def _run(M, N, K, fa, fb, shift=0, d_shift=0, odt=torch.float32, acc=False, seed=0):
    from nanotron_amd import _native as nt

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(seed)
    tab = {f: torch.tensor(O.decode_table(f), dtype=torch.float64, device=dev) for f in (O.E4M3, O.E5M2)}

    def operand(rows, fmt):
        buf = torch.zeros(rows * K + 64, dtype=torch.uint8, device=dev)
        q = buf[shift:shift + rows * K].view(rows, K)
        q.copy_(torch.randint(0, 256, (rows, K), generator=g, device=dev).to(torch.uint8))
        q[~torch.isfinite(tab[fmt][q.long()])] = 0x31   # NaN and Inf codes are covered elsewhere
        buf[shift + rows * K:] = 0x7f                   # a read past the operand that is not masked shows up as NaN
        return q

    a, b = operand(M, fa), operand(N, fb)
    one = torch.ones(1, device=dev)
    store = torch.zeros(M * N + 8, dtype=odt, device=dev)
    out = store[d_shift:d_shift + M * N].view(M, N)
    base = torch.randn(M, N, generator=g, device=dev) if acc else None
    if acc:
        out.copy_(base)
    print(f"M={M} N={N} K={K} fa={fa} fb={fb} shift={shift} d_shift={d_shift} {odt} acc={acc}", flush=True)
    nt.check(nt.lib.ntfp8_gemm(a.data_ptr(), 0 if fa == O.E4M3 else 1, one.data_ptr(), b.data_ptr(), 0 if fb == O.E4M3 else 1,
                               one.data_ptr(), out.data_ptr(), nt.TORCH_TO_NT[odt], M, N, K, int(acc), nt.stream_ptr(dev)), "gemm")
    a64, b64 = tab[fa][a.long()], tab[fb][b.long()]
    ref, mag = a64 @ b64.t(), a64.abs() @ b64.abs().t()
    if acc:
        ref, mag = ref + base.double(), mag + base.double().abs()
    slack = K * 2.0 ** -23 * mag
    if odt != torch.float32:
        slack = slack + ref.abs() * 2.0 ** -8 + 2.0 ** -126
    assert bool(((out.double() - ref).abs() <= slack).all())
    assert bool((store[M * N + d_shift:] == 0).all() and (store[:d_shift] == 0).all())


@pytest.mark.parametrize("fa,fb", [(O.E4M3, O.E4M3), (O.E5M2, O.E4M3), (O.E4M3, O.E5M2), (O.E5M2, O.E5M2)])
@pytest.mark.parametrize("K", [1, 15, 17, 127, 129, 383, 1021])
def test_edges_of_k(K, fa, fb):
    _run(65, 63, K, fa, fb, seed=K)


@pytest.mark.parametrize("M,N", [(1, 1), (64, 64), (65, 130), (7, 601), (2049, 2100)])   # the last: 128-wide tiles
@pytest.mark.parametrize("acc", [False, True])
def test_edges_of_the_tile(M, N, acc):
    _run(M, N, 141, O.E5M2, O.E4M3, acc=acc, seed=M)


@pytest.mark.parametrize("shift,d_shift,K,N", [(3, 0, 256, 96), (8, 1, 256, 96), (0, 1, 250, 64), (5, 3, 77, 40)])
@pytest.mark.parametrize("odt", [torch.float32, torch.bfloat16])
def test_views_that_start_anywhere(shift, d_shift, K, N, odt):
    _run(130, N, K, O.E4M3, O.E4M3, shift=shift, d_shift=d_shift, odt=odt, seed=shift)


# (M, N, K) around the lines between one output per thread and tiles: K below 40, 2^17 outputs, 40 * 2^16 products
@pytest.mark.parametrize("mnk", [(1, 1, 1), (255, 1, 17), (3, 86, 39), (3, 86, 41), (362, 362, 19), (363, 362, 19), (257, 255, 39), (259, 263, 39)])
@pytest.mark.parametrize("fa,fb", [(O.E4M3, O.E4M3), (O.E5M2, O.E4M3), (O.E4M3, O.E5M2), (O.E5M2, O.E5M2)])
def test_one_output_per_thread(mnk, fa, fb):
    _run(*mnk, fa, fb, seed=mnk[0])
    _run(*mnk, fa, fb, acc=True, seed=mnk[1])
    _run(*mnk, fa, fb, odt=torch.bfloat16, d_shift=1, seed=mnk[2])
    _run(*mnk, fa, fb, odt=torch.bfloat16, shift=1, seed=mnk[2])
