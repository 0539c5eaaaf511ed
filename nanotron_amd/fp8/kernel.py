from typing import Optional, Union

import torch

from nanotron_amd import _native as nt
from nanotron_amd.fp8.dtypes import DTypes
from nanotron_amd.fp8.tensor import DelayedScaling, FP8Tensor, _assemble


def _problem(a: FP8Tensor, b: FP8Tensor, out_code: int, accumulate_into=None, bt: bool = False, bias=None, at: bool = False):
    """The fields of one GEMM as csrc/hostcall.cpp takes them.  (A meta is a Python attribute of the FP8Tensor object; a
    copy made of a view does not carry it, so it is read here and the extension makes the copy.)"""
    ma, mb = a.fp8_meta, b.fp8_meta
    return (a, ma.dtype.code, ma.scale, b, mb.dtype.code, mb.scale, out_code, accumulate_into, bt, bias, at)


def _gemm_nt(a: FP8Tensor, b: FP8Tensor, out_dtype: torch.dtype, accumulate_into: Optional[torch.Tensor],
             bias: Optional[torch.Tensor] = None):
    """D[M,N] = A[M,K] . B[N,K]^T, descaled (te_gemm's TN form, src/nanotron/fp8/kernel.py:46-68); with `bias`
    [N] added to the descaled fp32 result before the single rounding (te_gemm's bias argument, which the
    reference leaves empty, kernel.py:29-32)."""
    return nt.host.gemm(*_problem(a, b, nt.TORCH_TO_NT[out_dtype], accumulate_into, False, bias))


def _gemm_nt_fp8(a: FP8Tensor, b: FP8Tensor, dtype: DTypes, state: Optional[DelayedScaling],
                 with_transpose: bool, bias: Optional[torch.Tensor] = None, bt: bool = False, at: bool = False) -> FP8Tensor:
    """FP8Tensor(_gemm_nt(a, b, float32), dtype, state=state, with_transpose=with_transpose), bit for bit, with the
    fp32 result never written to memory: the GEMM epilogue casts with the scale `state` holds from earlier steps, and
    the workgroup that finishes last turns max|result| into amax, history roll and next scale.

    The amax of a GEMM result is not known before the GEMM has run, so a step without a held scale (no `state`, or
    one that has not seen a usable amax yet) goes the long way: fp32 result, then the ordinary quantisation."""
    assert dtype.out_code is not None, f"{dtype} is not an FP8 format"
    if state is None or not state.known_initialised:
        hp = (_gemm_nt_batch([(a, b, torch.float32, None, True, None, at)])[0] if bt
              else _gemm_nt(a, b, torch.float32, None, bias))
        return FP8Tensor(hp, dtype, state=state, with_transpose=with_transpose)
    assert state.dtype == dtype, "delayed-scaling state was created for another format"
    assert not at or bt, "a transposed A operand is only read next to a transposed B operand"
    return _assemble(FP8Tensor, dtype, *nt.host.gemm_fp8(
        *_problem(a, b, dtype.out_code, None, bt, bias, at), state._buf, state.history_len, state.margin, with_transpose))


# Module switch: False makes every GEMM use materialised transposed copies (the reference's way, kernel.py:43-44).
READ_B_TRANSPOSED = True


def b_transposed_supported(M: int, N: int, K: int) -> bool:
    """Whether the library reads the B operand of D[M,N] = A[M,K] . B[N,K]^T from its transpose, a [K, N] tensor
    (`ntfp8_gemm_desc.b_transposed`): the condition stated in include/ntfp8.h."""
    return READ_B_TRANSPOSED and nt.host.b_transposed_supported(M, N, K)


# Module switch: False makes wgrad GEMMs take a materialised transpose of the output gradient (kernel.py:44).
READ_A_TRANSPOSED = True


def a_transposed_supported(M: int, N: int, K: int) -> bool:
    """Whether the library reads BOTH operands of D[M,N] = A[M,K] . B[N,K]^T from their transposes, [K, M] and [K, N]
    tensors (`ntfp8_gemm_desc.a_transposed` next to `b_transposed`): the wgrad form, dW = dY^T . X with dY[tokens, out]
    and X[tokens, in] as they are."""
    return READ_A_TRANSPOSED and M % 16 == 0 and b_transposed_supported(M, N, K)


def needs_transposed_copy(rows: int, cols: int, other: int = 4096) -> bool:
    """Whether a [rows, cols] fp8 tensor that a backward GEMM reduces over its rows (the weight in dgrad, the input in
    wgrad; src/nanotron/fp8/linear.py:104-109) should be quantised together with its transposed copy: only if the
    library cannot read it as it is.  `other` is the GEMM's third dimension (tokens for the weight, out_features
    for the input), assumed large when not known yet; a copy that turns out to be needed after all is made on demand."""
    return not b_transposed_supported(other, cols, rows)


def _gemm_nt_batch(problems):
    """Several independent `_gemm_nt` problems, given as tuples (a, b, out_dtype, accumulate_into[, b_transposed[,
    bias[, a_transposed]]]), in one call of the library: GEMMs with the same operand formats share launches.  With
    `b_transposed` the tensor `b` is the [K, N] transpose of the operand, with `a_transposed` the tensor `a` its [K, M]
    transpose.  Returns the outputs in order."""
    full = []
    for prob in problems:
        a, b, out_dtype, accumulate_into = prob[:4]
        full.append(_problem(a, b, nt.TORCH_TO_NT[out_dtype], accumulate_into, len(prob) > 4 and prob[4],
                             prob[5] if len(prob) > 5 else None, len(prob) > 6 and prob[6]))
    return nt.host.gemm_batch(full)


def _operands(mat_a: FP8Tensor, transpose_a: bool, mat_b: FP8Tensor, transpose_b: bool,
              accumulate_into: Optional[torch.Tensor] = None, allow_bt: bool = True):
    """(A, B, b_transposed, a_transposed) of the library's D = A . B^T for the reference's D = op_b(B) . op_a(A)
    (kernel.py:43-44).

    Where the reference transposes mat_a (tex.fp8_transpose, kernel.py:43) the library can read it as it is
    (`b_transposed`): that is taken when mat_a carries no transposed copy yet and the shape qualifies; otherwise the
    copy is used (and made, once, if it does not exist).  The same for mat_b (kernel.py:44, `a_transposed`), which the
    library serves next to an untransposed mat_a: the wgrad form."""
    form = nt.host.operand_form(mat_a, getattr(mat_a, "_transposed", None), transpose_a, mat_b, getattr(mat_b, "_transposed", None),
                                transpose_b, accumulate_into, allow_bt, READ_B_TRANSPOSED, READ_A_TRANSPOSED)
    assert hasattr(mat_a, "fp8_meta") and hasattr(mat_b, "fp8_meta"), "operands must be FP8Tensors"
    return (mat_b.transposed() if form & 1 else mat_b), (mat_a.transposed() if form & 2 else mat_a), bool(form & 4), bool(form & 8)


def fp8_matmul_pair(first: dict, second: dict):
    """Two independent `fp8_matmul_kernel` calls (keyword dictionaries of its arguments) issued together, e.g. the
    dgrad and wgrad of a layer (src/nanotron/fp8/linear.py:104-109 issues them one after the other).  Same
    results as two calls; the library lets the two GEMMs share kernel launches."""
    probs = []
    for kw in (first, second):
        acc = kw.get("accumulate_into")
        A, B, bt, at = _operands(kw["mat_a"], kw["transpose_a"], kw["mat_b"], kw["transpose_b"], acc)
        probs.append((A, B, torch.float32 if acc is not None else kw.get("out_dtype") or torch.float32, acc, bt, None, at))
    return _gemm_nt_batch(probs)


def fp8_matmul_kernel(
    mat_a: FP8Tensor,
    transpose_a: bool,
    mat_b: FP8Tensor,
    transpose_b: bool,
    use_split_accumulator: bool,
    *,
    out_dtype: Union[torch.dtype, DTypes, None] = None,
    accumulate_into: Optional[torch.Tensor] = None,
    out_state: Optional[DelayedScaling] = None,
    out_with_transpose: bool = False,
    bias: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """D = op_b(B) . op_a(A) * (1/scale_a)(1/scale_b), op_x(X) = X^T if transpose_x else X
    (reference: src/nanotron/fp8/kernel.py:9-70; the operator meaning follows from its fixed
    te_gemm(transa=True, transb=False) call on row-major tensors).  fp32 output unless `out_dtype`
    says otherwise (kernel.py:24,28).  The result has its true shape [rows of op_b(B), cols of
    op_a(A)], which equals the reference's allocation on the square shapes its tests use.

    `use_split_accumulator` selects cuBLASLt's slower, more accurate accumulation on Hopper; CDNA4
    matrix cores always accumulate in fp32, so it is accepted and ignored.
    `accumulate_into` (fp32, contiguous) receives D added in place before any rounding.
    `out_dtype=DTypes.FP8E4M3 / FP8E5M2` returns D as an FP8Tensor ("return an fp8 tensor as output", the TODO at
    src/nanotron/fp8/linear.py:63-64), quantised with the delayed-scaling state `out_state` in the GEMM's epilogue
    and, with `out_with_transpose`, carrying its transposed copy.
    `bias` (one value per column of D, fp32 / fp16 / bf16) is added to the descaled fp32 result before the single
    rounding to the output type: the bias argument of te_gemm that the reference leaves empty (kernel.py:29-32).
    For an fp32 output this equals `D + bias` bit for bit."""
    if isinstance(out_dtype, DTypes):
        assert accumulate_into is None, "an fp8 output cannot accumulate"
        # rows of D: the fp8 epilogue stores whole words of 4 rows' worth of the transposed copy
        rows = mat_b.as_subclass(torch.Tensor).shape[1 if transpose_b else 0]
        A, B, bt, at = _operands(mat_a, transpose_a, mat_b, transpose_b, None, allow_bt=bias is None and rows % 4 == 0)
        return _gemm_nt_fp8(A, B, out_dtype, out_state, out_with_transpose, bias, bt, at)
    A, B, bt, at = _operands(mat_a, transpose_a, mat_b, transpose_b, accumulate_into, allow_bt=bias is None)
    if bt:
        return _gemm_nt_batch([(A, B, out_dtype or torch.float32, accumulate_into, True, None, at)])[0]
    return _gemm_nt(A, B, out_dtype or torch.float32, accumulate_into, bias)
