"""The tile size that the library takes for a GEMM launch, for tests that have to know which kernel they reach."""
import ctypes

from nanotron_amd import _native as nt

F32, F16, BF16, OUT_E4M3 = 0, 1, 2, 3


def tiles(*problems, cus=256, copy=False):
    """(tile rows, tile columns, parts of a tile of the partial last round) of one launch of the problems (M, N, K, output code,
    form[, accumulate]), form 0 both operands K-contiguous, 1 B as its transpose, 2 both as their transposes, `copy`: with the transposed
    copy of an fp8 output; None where they do not go to the tile kernels together."""
    query = nt.lib.ntfp8_debug_gemm_tiles
    query.restype, query.argtypes = ctypes.c_int, [ctypes.POINTER(nt.GemmDesc), ctypes.c_int, ctypes.c_int] + [ctypes.POINTER(ctypes.c_int)] * 3
    d = (nt.GemmDesc * len(problems))()
    for g, (M, N, K, out, form, *acc) in zip(d, problems):
        g.M, g.N, g.K, g.d_dtype, g.b_transposed, g.a_transposed, g.accumulate = M, N, K, out, int(form > 0), int(form > 1), int(any(acc))
        g.D_t = 16 if copy else None
    m, n, parts = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    rc = query(d, len(problems), cus, ctypes.byref(m), ctypes.byref(n), ctypes.byref(parts))
    return (m.value, n.value, parts.value) if rc == 0 else None
