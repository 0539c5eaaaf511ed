"""Type arguments of the Transformer-Engine-shaped functions: plain numbers and enum members alike, looked up without running
any Python per argument (small calls are bound by the host)."""
import sys

import pytest

from nanotron_amd import tex_shim as tex
from nanotron_amd.fp8.dtypes import DType


@pytest.mark.parametrize("value", [*DType, *range(-1, 9)])
def test_fp8_types(value):
    want = {5: 0, 6: 1}.get(int(value))
    if want is None:
        with pytest.raises(RuntimeError, match="not an FP8 type"):
            tex._fmt(value)
    else:
        assert tex._fmt(value) == want


def test_a_type_costs_no_python_call():
    seen = []
    e4 = DType.kFloat8E4M3
    sys.setprofile(lambda frame, event, arg: seen.append(frame.f_code.co_name) if event == "call" else None)
    try:
        tex._fmt(e4)
    finally:
        sys.setprofile(None)
    assert seen == ["_fmt"]
