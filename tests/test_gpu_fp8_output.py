"""GPU parity of the fp8-output GEMM epilogue ("return an fp8 tensor as output", the TODO at
src/nanotron/fp8/linear.py:63-64).  The bar is bit-exactness on every output: the bytes (and their transposed
copy) equal the cast of the fp32 GEMM result, the amax equals that result's, and scale and amax history move as
in the stand-alone delayed-scaling quantisation.  Integer-valued operands, whose products sum exactly in any
order, tie the whole thing to the CPU oracle."""
import ctypes

import pytest
import torch

from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu

FMTS = [O.E4M3, O.E5M2]


def _dt(fmt):
    from nanotron_amd.fp8 import DTypes

    return DTypes.FP8E4M3 if fmt == O.E4M3 else DTypes.FP8E5M2


def from_bytes(q_cpu, scale, fmt):
    from nanotron_amd.fp8 import FP8Tensor
    from nanotron_amd.fp8.meta import FP8Meta

    t = torch.Tensor._make_subclass(FP8Tensor, q_cpu.cuda())
    t.fp8_meta = FP8Meta(torch.tensor(0.0, device="cuda"), torch.tensor(float(scale), dtype=torch.float32, device="cuda"),
                         _dt(fmt))
    return t


def _state_with_scale(fmt, scale, history_len=4, hist=None):
    """An initialised delayed-scaling state that holds `scale` for the next step."""
    from nanotron_amd.fp8 import DelayedScaling

    st = DelayedScaling(_dt(fmt), history_len=history_len, device="cuda")
    st._buf[0] = float(scale)
    if hist is not None:
        st._buf[1:] = torch.tensor(hist, dtype=torch.float32)
    st.initialised = True
    return st


def _clone_state(st):
    from nanotron_amd.fp8 import DelayedScaling

    c = DelayedScaling(st.dtype, history_len=st.history_len, margin=st.margin, device="cuda")
    c._buf.copy_(st._buf)
    c.initialised = st.initialised
    return c


def _same_f32(a, b):
    a, b = a.detach().float().cpu().reshape(-1), b.detach().float().cpu().reshape(-1)
    return bool(torch.all((a.view(torch.int32) == b.view(torch.int32)) | (a.isnan() & b.isnan())))


def _check_against_two_step(A, B, fo, st, with_transpose=True):
    """fused epilogue == fp32 GEMM followed by the delayed-scaling quantisation, on every output"""
    from nanotron_amd.fp8 import FP8Tensor
    from nanotron_amd.fp8.kernel import _gemm_nt, _gemm_nt_fp8

    st2 = _clone_state(st)
    got = _gemm_nt_fp8(A, B, _dt(fo), st, with_transpose)
    r = _gemm_nt(A, B, torch.float32, None)
    want = FP8Tensor(r, _dt(fo), state=st2, with_transpose=with_transpose)
    assert got.shape == r.shape and got.dtype == torch.uint8
    assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor))
    if with_transpose:
        assert torch.equal(got.transposed().as_subclass(torch.Tensor), want.transposed().as_subclass(torch.Tensor))
        assert torch.equal(got.transposed().as_subclass(torch.Tensor), got.as_subclass(torch.Tensor).t().contiguous())
    assert _same_f32(got.fp8_meta.amax, want.fp8_meta.amax)
    assert _same_f32(got.fp8_meta.scale, want.fp8_meta.scale)
    assert _same_f32(st._buf, st2._buf)
    from nanotron_amd import _native as nt

    ws = nt.workspace(torch.device("cuda", 0))
    assert int(ws.abs().sum().item()) == 0, "the reduction workspace must be left zeroed"
    return got, r


# shapes: big kernel whole tiles + half-tile tail, big kernel ragged edges, small kernel, small kernel ragged
# (N not a multiple of 16 / M not of 4), kernels of any K (K not a multiple of 16)
SHAPES = [(512, 768, 256), (2304, 2048, 384), (260, 400, 512), (1000, 144, 272), (128, 128, 128), (64, 48, 32),
          (130, 250, 272), (131, 200, 256), (33, 17, 96), (5, 3, 7), (1, 1, 1), (200, 36, 1040)]


@pytest.mark.parametrize("mnk", SHAPES)
@pytest.mark.parametrize("fo", FMTS)
def test_integer_operands_match_the_oracle_bit_for_bit(mnk, fo):
    M, N, K = mnk
    g = torch.Generator().manual_seed(M * 7 + N * 3 + K)
    a = torch.randint(-4, 5, (M, K), generator=g).float()
    b = torch.randint(-4, 5, (N, K), generator=g).float()
    one = torch.tensor(1.0)
    fa, fb = O.E4M3, (O.E5M2 if (M + N) % 2 else O.E4M3)
    aq, bq = O.cast_to_fp8(a, one, fa), O.cast_to_fp8(b, one, fb)
    r_ref = O.gemm_nt(aq, fa, torch.tensor(2.0), bq, fb, torch.tensor(4.0))   # exact: integers / 8
    assert torch.equal(r_ref, (a.double() @ b.double().t()).float() / 8)
    A, B = from_bytes(aq, 2.0, fa), from_bytes(bq, 4.0, fb)
    for scale in (0.25, 8.0, 4096.0):   # the last one saturates e4m3 for the larger sums
        st = _state_with_scale(fo, scale, hist=[3.0, 0.5, 0.0, 0.0])
        got, r = _check_against_two_step(A, B, fo, st)
        assert torch.equal(r.cpu(), r_ref)
        want = O.cast_to_fp8(r_ref, torch.tensor(scale), fo)
        assert torch.equal(got.as_subclass(torch.Tensor).cpu(), want)
        amax = r_ref.abs().max()
        assert _same_f32(got.fp8_meta.amax, amax)
        # history rolled, newest first; next scale from the history's maximum
        assert _same_f32(st.amax_history, torch.tensor([float(amax), 3.0, 0.5, 0.0]))
        nxt = O.update_scaling_factor(torch.maximum(amax, torch.tensor(3.0)), torch.tensor(scale), fo)
        assert _same_f32(st.scale, nxt)


@pytest.mark.parametrize("fa,fb", [(O.E4M3, O.E4M3), (O.E5M2, O.E4M3), (O.E4M3, O.E5M2)])
@pytest.mark.parametrize("fo", FMTS)
@pytest.mark.parametrize("mnk", [(512, 768, 256), (2304, 2048, 384), (260, 400, 512), (96, 80, 128), (128, 256, 4096)])
def test_random_operands_equal_cast_of_the_fp32_result(fa, fb, fo, mnk):
    from nanotron_amd.fp8 import FP8Tensor

    M, N, K = mnk
    x = O.normal_tensor(M + 1, (M, K), 1.0, torch.bfloat16)
    w = O.normal_tensor(N + 2, (N, K), 0.05, torch.bfloat16)
    A = FP8Tensor(x.cuda(), _dt(fa))
    B = FP8Tensor(w.cuda(), _dt(fb))
    st = _state_with_scale(fo, 16.0, history_len=16)
    for _ in range(3):   # the scale moves after the first step
        got, r = _check_against_two_step(A, B, fo, st, with_transpose=True)
    # and against the oracle's arithmetic: dequantised, within the GEMM tolerance plus one fp8 rounding
    xq, wq = O.quantise_current(x, fa), O.quantise_current(w, fb)
    r_ref = O.gemm_nt(xq.q, fa, xq.scale, wq.q, fb, wq.scale)
    assert O.rel_l2(r.cpu(), r_ref) <= 1e-3
    deq = O.upcast(got.as_subclass(torch.Tensor).cpu(), fo) / got.fp8_meta.scale.cpu()
    assert O.rel_l2(deq, r_ref) <= (0.04 if fo == O.E4M3 else 0.08)


@pytest.mark.parametrize("mnk", [(512, 768, 256), (96, 80, 128), (33, 17, 100)])   # big, small, any K
@pytest.mark.parametrize("fo", FMTS)
def test_nan_inf_and_degenerate_scales(mnk, fo):
    M, N, K = mnk
    g = torch.Generator().manual_seed(5)
    a = torch.randint(-4, 5, (M, K), generator=g).float()
    b = torch.randint(-4, 5, (N, K), generator=g).float()
    one = torch.tensor(1.0)
    aq, bq = O.cast_to_fp8(a, one, O.E5M2), O.cast_to_fp8(b, one, O.E4M3)
    aq[3, 5] = 0x7C    # +Inf (e5m2): row 3 of the result is +-Inf or NaN
    aq[M - 1, 0] = 0xFE    # -NaN (e5m2): the last row is NaN
    bq[1, 2] = 0x7F    # NaN (e4m3): column 1 is NaN
    A, B = from_bytes(aq, 1.0, O.E5M2), from_bytes(bq, 1.0, O.E4M3)
    st = _state_with_scale(fo, 2.0)
    before = st._buf.clone()
    got, r = _check_against_two_step(A, B, fo, st)
    q = got.as_subclass(torch.Tensor).cpu()
    rc = r.cpu()
    assert rc.isnan().any() and rc.isinf().any()
    assert torch.equal(q, O.cast_to_fp8(rc, torch.tensor(2.0), fo))
    assert bool(((q[rc.isnan()] & 0x7F) == 0x7F).all())                     # NaN -> sign | 0x7F
    fmax_code = 0x7E if fo == O.E4M3 else 0x7B
    assert bool(((q[rc.isinf()] & 0x7F) == fmax_code).all())                 # +-Inf saturate
    assert torch.isnan(got.fp8_meta.amax).item()                              # NaN-propagating amax
    assert _same_f32(st.scale, before[0])                                     # ... which holds the scale
    # degenerate scales: every product may be NaN (0 * Inf), the patching runs on all of them
    for s in (0.0, float("inf")):
        st = _state_with_scale(fo, s)
        got, r = _check_against_two_step(A, B, fo, st)
        assert torch.equal(got.as_subclass(torch.Tensor).cpu(), O.cast_to_fp8(r.cpu(), torch.tensor(s), fo))


def test_first_step_without_a_held_scale_uses_current_scaling():
    from nanotron_amd.fp8 import DelayedScaling, FP8Tensor
    from nanotron_amd.fp8.kernel import _gemm_nt, fp8_matmul_kernel

    x = O.normal_tensor(1, (384, 256), 1.0, torch.bfloat16)
    w = O.normal_tensor(2, (512, 256), 0.05, torch.bfloat16)
    X, W = FP8Tensor(x.cuda(), _dt(O.E4M3)), FP8Tensor(w.cuda(), _dt(O.E4M3), with_transpose=True)
    st = DelayedScaling(_dt(O.E4M3), history_len=4, device="cuda")
    st2 = _clone_state(st)
    r = _gemm_nt(X, W, torch.float32, None)
    for step in range(3):   # step 0: no scale held yet; steps 1, 2: the fused epilogue
        got = fp8_matmul_kernel(W, True, X, False, False, out_dtype=_dt(O.E4M3), out_state=st, out_with_transpose=True)
        want = FP8Tensor(r, _dt(O.E4M3), state=st2, with_transpose=True)
        assert st.initialised
        assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor))
        assert torch.equal(got.transposed().as_subclass(torch.Tensor), want.transposed().as_subclass(torch.Tensor))
        assert _same_f32(st._buf, st2._buf) and _same_f32(got.fp8_meta.scale, want.fp8_meta.scale)
    # no state at all: current scaling every time
    got = fp8_matmul_kernel(W, True, X, False, False, out_dtype=_dt(O.E5M2))
    want = FP8Tensor(r, _dt(O.E5M2))
    assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor))


def test_two_linears_chained_through_an_fp8_activation():
    from nanotron_amd.fp8 import DTypes, FP8Linear, FP8Parameter, FP8Tensor

    T, H, I = 320, 256, 384
    w1 = O.normal_tensor(11, (I, H), 0.05, torch.float32)
    w2 = O.normal_tensor(12, (H, I), 0.05, torch.float32)
    first = FP8Linear(H, I, bias=False, device="cuda", out_dtype=DTypes.FP8E4M3, delayed_scaling=True, amax_history_len=4,
                      fp8_output_transpose=True)
    second = FP8Linear(I, H, bias=False, device="cuda", delayed_scaling=True, amax_history_len=4)
    plain = FP8Linear(H, I, bias=False, device="cuda", delayed_scaling=True, amax_history_len=4)   # fp32 output twin
    for lin, w in ((first, w1), (second, w2), (plain, w1)):
        lin.weight = FP8Parameter(w.cuda(), DTypes.FP8E4M3)
    ref_state = _clone_state(first.scaling["output"])
    for step in range(3):
        x = O.normal_tensor(20 + step, (T, H), 1.0 + step, torch.bfloat16).cuda()
        with torch.no_grad():
            h = first(x)
            y = second(h)
            h32 = plain(x)
        assert isinstance(h, FP8Tensor) and h.shape == (T, I) and not h.requires_grad
        want_h = FP8Tensor(h32, DTypes.FP8E4M3, state=ref_state, with_transpose=True)
        assert torch.equal(h.as_subclass(torch.Tensor), want_h.as_subclass(torch.Tensor))
        assert _same_f32(first.scaling["output"]._buf, ref_state._buf)
        # the second layer consumed the bytes as they are (no re-quantisation): oracle on the same bytes
        hq = O.Quantised(h.as_subclass(torch.Tensor).cpu(), h.fp8_meta.amax.cpu(), h.fp8_meta.scale.cpu(), O.E4M3)
        wq = O.quantise_current(w2, O.E4M3)
        assert O.rel_l2(y.cpu(), O.linear_forward(hq, wq)) <= 1e-3
    # a bias is allowed with an fp8 output: it is added in the epilogue, before the cast (tests/test_gpu_extensions.py)
    assert FP8Linear(H, I, bias=True, device="cuda", out_dtype=DTypes.FP8E4M3).bias is not None
    with pytest.raises(ValueError):
        FP8Linear(H, I, bias=False, device="cuda", out_dtype=DTypes.KFLOAT16)
    assert "fp8_state.output" in first.state_dict()


def test_gradient_of_an_fp8_activation_goes_back_as_fp8_bytes():
    """Backward of a chain FP8Linear(out fp8) -> FP8Linear: once the producer's output-gradient role holds a scale, the
    consumer's dgrad epilogue writes dX as e5m2 bytes under that role (the TODO at src/nanotron/fp8/linear.py:63-64,
    backward direction) and autograd only carries a placeholder.  The bytes, the scale used and the role's state must
    equal the quantisation of the fp32 dgrad result under the same role; the producer's gradients are then checked
    against the oracle on those bytes.  With a second consumer of the same activation both send high-precision gradients."""
    from nanotron_amd.fp8 import DTypes, FP8Linear, FP8Parameter, FP8Tensor
    from nanotron_amd.fp8.kernel import fp8_matmul_kernel

    T, H, I = 384, 256, 512
    w1 = O.normal_tensor(51, (I, H), 0.05, torch.float32)
    w2 = O.normal_tensor(52, (H, I), 0.05, torch.float32)
    first = FP8Linear(H, I, bias=False, device="cuda", out_dtype=DTypes.FP8E4M3, delayed_scaling=True, amax_history_len=4)
    second = FP8Linear(I, H, bias=False, device="cuda", delayed_scaling=True, amax_history_len=4, out_dtype=torch.bfloat16)
    for lin, w in ((first, w1), (second, w2)):
        lin.weight = FP8Parameter(w.cuda(), DTypes.FP8E4M3)
        lin.keep_quantised_grad = True
    for step in range(4):
        x = O.normal_tensor(60 + step, (T, H), 1.0 + 0.5 * step, torch.bfloat16).cuda().requires_grad_(True)
        gy = O.normal_tensor(70 + step, (T, H), 1e-3 * (1 + step), torch.bfloat16).cuda()
        role = first.scaling["output_grad"]
        fp8_path = role.initialised   # (reads the flag: from the second step on)
        before = _clone_state(role)
        h = first(x)
        y = second(h)
        y.backward(gy)
        got = first.quantised_grad_output          # what the producer's backward GEMMs read
        assert isinstance(got, FP8Tensor) and got.fp8_meta.dtype == DTypes.FP8E5M2 and tuple(got.shape) == (T, I)
        # the fp32 dgrad of the consumer on the operands it used, quantised under the producer's role as it stood
        dx32 = fp8_matmul_kernel(mat_a=second.weight.data, transpose_a=False, mat_b=second.quantised_grad_output,
                                 transpose_b=False, use_split_accumulator=True)
        if fp8_path:
            want = FP8Tensor(dx32, DTypes.FP8E5M2, state=before)
            assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor)), step
            assert _same_f32(got.fp8_meta.scale, want.fp8_meta.scale) and _same_f32(got.fp8_meta.amax, want.fp8_meta.amax), step
            assert _same_f32(role._buf, before._buf), step
        else:
            # through the high-precision handle: rounded to its type (the producer's master-weight type), then quantised
            want = FP8Tensor(dx32.to(h._grad_handle.dtype), DTypes.FP8E5M2, state=before)
            assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor)), step
        # the producer's own gradients from those bytes, against the oracle
        gq = O.Quantised(got.as_subclass(torch.Tensor).cpu(), got.fp8_meta.amax.cpu(), got.fp8_meta.scale.cpu(), O.E5M2)
        wq = O.Quantised(first.weight.data.as_subclass(torch.Tensor).cpu(), first.weight.data.fp8_meta.amax.cpu(),
                         first.weight.data.fp8_meta.scale.cpu(), O.E4M3)
        assert O.rel_l2(x.grad.float().cpu(), O.linear_dgrad(gq, wq).to(torch.bfloat16).float()) <= 1e-3, step
        assert first.weight.grad is not None and second.weight.grad is not None
    # two consumers of one fp8 activation: fp8 contributions cannot be summed, so both send high-precision gradients that
    # autograd sums on the handle, and nothing goes back as fp8
    third = FP8Linear(I, H, bias=False, device="cuda", delayed_scaling=True, out_dtype=torch.bfloat16)
    x = O.normal_tensor(99, (T, H), 1.0, torch.bfloat16).cuda().requires_grad_(True)
    sent = (second.fp8_grad_inputs_sent, third.fp8_grad_inputs_sent)
    for _ in range(3):   # (these gradients are far larger than the steps' above: let the delayed scales of both levels settle)
        x.grad = None
        h = first(x)
        (second(h).float().sum() + third(h).float().sum()).backward()
    assert (second.fp8_grad_inputs_sent, third.fp8_grad_inputs_sent) == sent
    both = x.grad.float().clone()
    assert bool(torch.isfinite(both).all()) and float(both.abs().max()) > 0
    # ... the same as with the fp8 hand-over switched off by hand
    second.fp8_grad_input = third.fp8_grad_input = False
    for lin in (first, second, third):
        lin.train(False)     # evaluation mode: the scaling roles stay as they are, so the two passes are comparable
    x.grad = None
    h = first(x)
    (second(h).float().sum() + third(h).float().sum()).backward()
    by_hand = x.grad.float().clone()
    second.fp8_grad_input = third.fp8_grad_input = True
    x.grad = None
    h = first(x)
    (second(h).float().sum() + third(h).float().sum()).backward()
    assert torch.equal(x.grad.float(), by_hand)
    # one consumer again: back to fp8
    for lin in (first, second, third):
        lin.train(True)
    h = first(x)
    second(h).float().sum().backward()
    assert second.fp8_grad_inputs_sent == sent[0] + 1


def test_fp8_activation_and_gradient_between_the_benchmark_mlp_linears_at_full_size():
    """The fp8 hand-over in both directions at the benchmark's size: up projection 4096 -> 14336 with an e4m3 output,
    down projection 14336 -> 4096, 4096 tokens, bf16 master weights, three delayed-scaling steps.  Forward: the bytes of
    the activation equal the delayed-scaling quantisation of the fp32 result of the same GEMM.  Backward: the e5m2 bytes
    the down projection's dgrad epilogue leaves for the up projection (896 whole tiles and a half-tile tail, operands
    read untransposed) equal the quantisation of its fp32 dgrad result under the same role; the up projection's own
    gradients are compared with the oracle on sampled rows."""
    from nanotron_amd.fp8 import DTypes, FP8Linear, FP8Parameter, FP8Tensor
    from nanotron_amd.fp8.kernel import fp8_matmul_kernel

    T, H, I = 4096, 4096, 14336
    g = torch.Generator(device="cuda").manual_seed(11)
    up = FP8Linear(H, I, bias=False, device="cuda", dtype=torch.bfloat16, out_dtype=DTypes.FP8E4M3, delayed_scaling=True)
    down = FP8Linear(I, H, bias=False, device="cuda", dtype=torch.bfloat16, out_dtype=torch.bfloat16, delayed_scaling=True)
    up.weight = FP8Parameter((torch.randn(I, H, generator=g, device="cuda") * 0.02).to(torch.bfloat16), DTypes.FP8E4M3)
    down.weight = FP8Parameter((torch.randn(H, I, generator=g, device="cuda") * 0.02).to(torch.bfloat16), DTypes.FP8E4M3)
    up.keep_quantised_grad = down.keep_quantised_grad = True
    rows = torch.arange(0, T, 67, device="cuda")[:48]
    sent = 0
    for step in range(3):
        x = (torch.randn(T, H, generator=g, device="cuda") * (1.0 + 0.5 * step)).to(torch.bfloat16).requires_grad_(True)
        gy = (torch.randn(T, H, generator=g, device="cuda") * 1e-3 * (1 + step)).to(torch.bfloat16)
        out_role, grad_role = up.scaling["output"], up.scaling["output_grad"]
        bwd_fused = grad_role.initialised
        out_before, grad_before = _clone_state(out_role), _clone_state(grad_role)
        h = up(x)
        assert isinstance(h, FP8Tensor) and tuple(h.shape) == (T, I)
        # forward: the activation against the long way on the operands the layer used (a role without a scale yet
        # quantises with current scaling either way)
        xq = h._grad_handle.grad_fn.saved_tensors[0]
        r32 = fp8_matmul_kernel(mat_a=up.weight.data, transpose_a=True, mat_b=xq, transpose_b=False, use_split_accumulator=False)
        want_h = FP8Tensor(r32, DTypes.FP8E4M3, state=out_before)
        assert torch.equal(h.as_subclass(torch.Tensor), want_h.as_subclass(torch.Tensor)), step
        assert _same_f32(h.fp8_meta.scale, want_h.fp8_meta.scale) and _same_f32(out_role._buf, out_before._buf), step
        del r32, want_h
        y = down(h)
        y.backward(gy)
        dx32 = fp8_matmul_kernel(mat_a=down.weight.data, transpose_a=False, mat_b=down.quantised_grad_output,
                                 transpose_b=False, use_split_accumulator=True)
        got = up.quantised_grad_output
        assert isinstance(got, FP8Tensor) and got.fp8_meta.dtype == DTypes.FP8E5M2 and tuple(got.shape) == (T, I)
        if bwd_fused:
            sent += 1
            assert down.fp8_grad_inputs_sent == sent
            want = FP8Tensor(dx32, DTypes.FP8E5M2, state=grad_before)
            assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor)), step
            assert _same_f32(got.fp8_meta.scale, want.fp8_meta.scale) and _same_f32(got.fp8_meta.amax, want.fp8_meta.amax), step
            assert _same_f32(grad_role._buf, grad_before._buf), step
        else:
            want = FP8Tensor(dx32.to(h._grad_handle.dtype), DTypes.FP8E5M2, state=grad_before)
            assert torch.equal(got.as_subclass(torch.Tensor), want.as_subclass(torch.Tensor)), step
        # the up projection's gradients from those bytes, against the oracle on sampled rows of dX and of dW
        gq = O.Quantised(got.as_subclass(torch.Tensor)[rows].cpu(), got.fp8_meta.amax.cpu(), got.fp8_meta.scale.cpu(), O.E5M2)
        wq = O.Quantised(up.weight.data.as_subclass(torch.Tensor).cpu(), up.weight.data.fp8_meta.amax.cpu(),
                         up.weight.data.fp8_meta.scale.cpu(), O.E4M3)
        assert O.rel_l2(x.grad[rows].float().cpu(), O.linear_dgrad(gq, wq, torch.bfloat16).float()) <= 1e-3, step
        assert up.weight.main_grad is not None and bool(torch.isfinite(up.weight.main_grad).all())
    assert sent >= 1


def test_an_fp8_activation_that_lost_its_gradient_handle_is_refused():
    """The gradient of an fp8 activation travels through the `_grad_handle` attribute of the object the producing layer
    returned.  A tensor derived from it (here: the same bytes re-wrapped, meta carried over) has no handle; consuming it
    with autograd on would leave the producer without any gradient, silently, so the consumer refuses."""
    from nanotron_amd.fp8 import DTypes, FP8Linear, FP8Tensor

    first = FP8Linear(256, 384, bias=False, device="cuda", out_dtype=DTypes.FP8E4M3, delayed_scaling=True)
    second = FP8Linear(384, 256, bias=False, device="cuda", delayed_scaling=True)
    x = O.normal_tensor(31, (320, 256), 1.0, torch.bfloat16).cuda().requires_grad_(True)
    for _ in range(2):   # the output role holds a scale from the second step on (the epilogue path)
        h = first(x)
        assert h._grad_handle is not None and h.fp8_meta.from_fp8_linear
        second(h).float().sum().backward()   # the object itself: fine, the producer gets its gradients
        assert x.grad is not None and first.weight.grad is not None
    h = first(x)
    derived = torch.Tensor._make_subclass(FP8Tensor, h.as_subclass(torch.Tensor).view(320, 384))
    derived.fp8_meta = h.fp8_meta
    with pytest.raises(RuntimeError, match="gradient handle"):
        second(derived)
    with torch.no_grad():   # without autograd there is nothing to lose
        second(derived)
    derived._grad_handle = h._grad_handle   # carried over by the caller: accepted
    second(derived).float().sum().backward()


@pytest.mark.parametrize("fo", FMTS)
@pytest.mark.parametrize("form", ["dgrad", "wgrad"])
@pytest.mark.parametrize("shape", [(512, 384, 640), (4096, 1024, 2048), (272, 400, 288)])
def test_fp8_output_with_operands_read_untransposed_equals_the_materialised_transposes(fo, form, shape):
    """An fp8 output next to `b_transposed` (dgrad form) and `a_transposed` + `b_transposed` (wgrad form): bytes,
    transposed bytes, amax, scale and history equal those of the same GEMM on transposed copies, bit for bit, and both
    equal the two-step form (fp32 GEMM, then the delayed-scaling cast)."""
    import nanotron_amd.fp8.kernel as K
    from nanotron_amd.fp8 import FP8Tensor
    from nanotron_amd.fp8.kernel import fp8_matmul_kernel

    T, n_out, k_in = shape
    gy = FP8Tensor(O.normal_tensor(11, (T, n_out), 1e-2, torch.bfloat16).cuda(), _dt(O.E5M2))
    w = FP8Tensor(O.normal_tensor(12, (n_out, k_in), 0.05, torch.bfloat16).cuda(), _dt(O.E4M3))
    x = FP8Tensor(O.normal_tensor(13, (T, k_in), 1.0, torch.bfloat16).cuda(), _dt(O.E4M3))
    if form == "dgrad":     # dX[T, k_in] = dY . W        (linear.py:104-106)
        args = dict(mat_a=w, transpose_a=False, mat_b=gy, transpose_b=False)
    else:                   # dW[n_out, k_in] = dY^T . X  (linear.py:107-109)
        args = dict(mat_a=x, transpose_a=False, mat_b=gy, transpose_b=True)
    st0 = _state_with_scale(fo, 64.0, history_len=4, hist=[0.5, 0.25, 2.0, 1.0])
    res = {}
    for mode in ("as_is", "copies"):
        K.READ_B_TRANSPOSED = K.READ_A_TRANSPOSED = mode == "as_is"
        try:
            for t in (gy, w, x):
                t._transposed = None
            st = _clone_state(st0)
            A, B, bt, at = K._operands(args["mat_a"], False, args["mat_b"], args["transpose_b"], None)
            assert (bt, at) == ((True, form == "wgrad") if mode == "as_is" else (False, False))
            for t in (gy, w, x):
                t._transposed = None
            out = fp8_matmul_kernel(**args, use_split_accumulator=False, out_dtype=_dt(fo), out_state=st, out_with_transpose=True)
            res[mode] = (out, st)
        finally:
            K.READ_B_TRANSPOSED = K.READ_A_TRANSPOSED = True
    (o1, s1), (o2, s2) = res["as_is"], res["copies"]
    assert torch.equal(o1.as_subclass(torch.Tensor), o2.as_subclass(torch.Tensor))
    assert torch.equal(o1._transposed.as_subclass(torch.Tensor), o2._transposed.as_subclass(torch.Tensor))
    assert torch.equal(o1._transposed.as_subclass(torch.Tensor), o1.as_subclass(torch.Tensor).t().contiguous())
    assert _same_f32(o1.fp8_meta.amax, o2.fp8_meta.amax) and _same_f32(o1.fp8_meta.scale, o2.fp8_meta.scale)
    assert _same_f32(s1._buf, s2._buf)
    # the two-step form on the fp32 result of the same kernel
    hp = fp8_matmul_kernel(**args, use_split_accumulator=False)
    two = FP8Tensor(hp, _dt(fo), state=_clone_state(st0))
    assert torch.equal(o1.as_subclass(torch.Tensor), two.as_subclass(torch.Tensor))
    assert _same_f32(o1.fp8_meta.amax, two.fp8_meta.amax)


def test_batch_mixes_fp8_and_plain_outputs_and_rejects_bad_requests():
    from nanotron_amd import _native as nt
    from nanotron_amd.fp8 import FP8Tensor

    dev = torch.device("cuda", 0)
    x = FP8Tensor(O.normal_tensor(1, (512, 256), 1.0, torch.bfloat16).cuda(), _dt(O.E4M3))
    w1 = FP8Tensor(O.normal_tensor(2, (768, 256), 0.05, torch.bfloat16).cuda(), _dt(O.E4M3))
    w2 = FP8Tensor(O.normal_tensor(3, (1024, 256), 0.05, torch.bfloat16).cuda(), _dt(O.E4M3))
    scale = torch.tensor([8.0, 32.0], device=dev)
    ws = torch.zeros(2, nt.WORKSPACE_BYTES // 4, dtype=torch.int32, device=dev)
    outs = [torch.empty(512, 768, dtype=torch.uint8, device=dev), torch.empty(512, 1024, dtype=torch.uint8, device=dev),
            torch.empty(512, 768, dtype=torch.bfloat16, device=dev)]
    out_t = torch.empty(1024, 512, dtype=torch.uint8, device=dev)
    st = nt.stream_ptr(dev)

    def desc(w, out, d_dtype, i=None, t=None, acc=0):
        d = nt.GemmDesc()
        d.A, d.scale_a, d.B, d.scale_b, d.D = (x.data_ptr(), x.fp8_meta.scale.data_ptr(), w.data_ptr(),
                                               w.fp8_meta.scale.data_ptr(), out.data_ptr())
        d.M, d.N, d.K = 512, w.shape[0], 256
        d.fmt_a, d.fmt_b, d.d_dtype, d.accumulate = nt.E4M3, nt.E4M3, d_dtype, acc
        if i is not None:
            d.scale_d, d.amax_workspace = scale[i:].data_ptr(), ws[i].data_ptr()
            d.D_t = nt.ptr(t)
        return d

    batch = (nt.GemmDesc * 3)(desc(w1, outs[0], nt.OUT_E4M3, 0), desc(w2, outs[1], nt.OUT_E5M2, 1, out_t),
                              desc(w1, outs[2], nt.BF16))
    nt.check(nt.lib.ntfp8_gemm_batch(batch, 3, st), "ntfp8_gemm_batch")
    from nanotron_amd.fp8.kernel import _gemm_nt
    from nanotron_amd.fp8.tensor import cast_with_scale

    r1, r2 = _gemm_nt(x, w1, torch.float32, None), _gemm_nt(x, w2, torch.float32, None)
    assert torch.equal(outs[0], cast_with_scale(r1, scale[0], _dt(O.E4M3)).as_subclass(torch.Tensor))
    assert torch.equal(outs[1], cast_with_scale(r2, scale[1], _dt(O.E5M2)).as_subclass(torch.Tensor))
    assert torch.equal(out_t, outs[1].t().contiguous())
    assert torch.equal(outs[2], _gemm_nt(x, w1, torch.bfloat16, None))
    amax = torch.zeros(2, device=dev)
    used = torch.zeros(2, device=dev)
    state = scale.clone()
    for i, r in enumerate((r1, r2)):
        nt.check(nt.lib.ntfp8_amax_finalize(ws[i].data_ptr(), i, 0, state[i:].data_ptr(), None, 0, amax[i:].data_ptr(),
                                            used[i:].data_ptr(), st), "ntfp8_amax_finalize")
        assert _same_f32(amax[i], r.abs().max()) and _same_f32(used[i], scale[i])
    assert torch.equal(state, scale) and int(ws.abs().sum().item()) == 0   # no history: the scale is left alone

    # refusals
    codes = {nt.strerror(c): c for c in range(-8, 1)}
    bad = (nt.GemmDesc * 1)(desc(w1, outs[0], nt.OUT_E4M3, 0, acc=1))
    assert nt.lib.ntfp8_gemm_batch(bad, 1, st) == codes["request not supported"]
    d = desc(w1, outs[0], nt.OUT_E4M3, 0)
    d.scale_d = None
    assert nt.lib.ntfp8_gemm_batch((nt.GemmDesc * 1)(d), 1, st) == codes["a required pointer is NULL"]
    d = desc(w1, outs[0], nt.OUT_E4M3, 0)
    d.D_t = outs[0].data_ptr() + 16
    assert nt.lib.ntfp8_gemm_batch((nt.GemmDesc * 1)(d), 1, st) == codes["an output overlaps an input or another output"]
    two = (nt.GemmDesc * 2)(desc(w1, outs[0], nt.OUT_E4M3, 0), desc(w2, outs[1], nt.OUT_E5M2, 0))   # shared amax slots
    assert nt.lib.ntfp8_gemm_batch(two, 2, st) == codes["an output overlaps an input or another output"]
    rc = nt.lib.ntfp8_gemm(x.data_ptr(), nt.E4M3, x.fp8_meta.scale.data_ptr(), w1.data_ptr(), nt.E4M3,
                           w1.fp8_meta.scale.data_ptr(), outs[0].data_ptr(), nt.OUT_E4M3, 512, 768, 256, 0, st)
    assert rc == codes["request not supported"]
    assert nt.lib.ntfp8_amax_finalize(ws[0].data_ptr(), 0, 0, state.data_ptr(), state.data_ptr(), 0, amax.data_ptr(), None,
                                      st) == codes["size, history length or margin out of range"]
    assert nt.lib.ntfp8_amax_finalize(None, 0, 0, state.data_ptr(), None, 0, amax.data_ptr(), None, st) == codes["a required pointer is NULL"]
    torch.cuda.synchronize()
    assert ctypes.sizeof(nt.GemmDesc) == 136


def test_fp8_output_chain_replayed_as_a_graph_matches_eager():
    """GEMM epilogue atomics into the workspace, the one-wave bookkeeping kernel that zeroes it again and nothing
    allocated in between: the forward of two chained layers can be captured and replayed; three replays with fresh
    inputs and unrelated eager work in between, against an eager twin, bit for bit including the scaling state."""
    from nanotron_amd.fp8 import DTypes, FP8Linear

    def build():
        torch.manual_seed(5)
        return (FP8Linear(256, 512, bias=False, device="cuda", out_dtype=DTypes.FP8E4M3, delayed_scaling=True, amax_history_len=4),
                FP8Linear(512, 256, bias=False, device="cuda", out_dtype=torch.bfloat16, delayed_scaling=True, amax_history_len=4))

    def fwd(layers, x):
        with torch.no_grad():
            return layers[1](layers[0](x))

    def inputs(i):
        return O.normal_tensor(700 + i, (384, 256), 1.0 + 0.2 * i, torch.bfloat16).cuda()

    g_layers, e_layers = build(), build()
    sx = torch.zeros(384, 256, dtype=torch.bfloat16, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):   # warm-up on the capture stream: every scaling role holds a scale afterwards
        for i in range(2):
            sx.copy_(inputs(i))
            fwd(g_layers, sx)
    torch.cuda.current_stream().wait_stream(side)
    for i in range(2):
        fwd(e_layers, inputs(i))
    torch.cuda.synchronize()
    assert g_layers[0].scaling["output"].initialised
    graph = torch.cuda.CUDAGraph()
    sx.copy_(inputs(2))
    with torch.cuda.graph(graph):
        sy = fwd(g_layers, sx)
    for i in range(2, 5):
        x = inputs(i)
        sx.copy_(x)
        graph.replay()
        ye = fwd(e_layers, x)
        _ = (ye.float() @ ye.float().t()).sum().item()   # unrelated eager work and a synchronisation in between
        assert torch.equal(sy, ye)
        for a, b in zip(g_layers, e_layers):
            for role in a.scaling:
                assert _same_f32(a.scaling[role]._buf, b.scaling[role]._buf), role
