"""Format tags, same names and values as the reference (src/nanotron/fp8/dtypes.py:4-7), plus the
stand-in for Transformer Engine's `tex.DType` enum that `FP8Meta.te_dtype` returns."""
from enum import Enum, IntEnum, auto


class DTypes(Enum):
    FP8E4M3 = auto()
    FP8E5M2 = auto()
    KFLOAT16 = auto()


# The native library's codes of a format (storage, and as a GEMM's output type), as plain attributes: a dictionary keyed by
# enum members hashes in Python on every look-up.  KFLOAT16 is no FP8 format.
for _member, _code, _out_code in ((DTypes.FP8E4M3, 0, 3), (DTypes.FP8E5M2, 1, 4), (DTypes.KFLOAT16, None, None)):
    _member.code, _member.out_code = _code, _out_code


class DType(IntEnum):
    """Element types understood by the native library; member names follow tex.DType
    (used at src/nanotron/fp8/tensor.py:39-55)."""

    kByte = 0
    kInt32 = 1
    kFloat32 = 2
    kFloat16 = 3
    kBFloat16 = 4
    kFloat8E4M3 = 5
    kFloat8E5M2 = 6
