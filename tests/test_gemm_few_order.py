"""`gemm_few_kernel` waits for a slot of its pipeline by counting the loads requested since, so in the generated code the loads
of a slot have to be older than those of the next: the opening requests of every instantiation, slot by slot."""
import os
import re
import subprocess

import pytest

from nanotron_amd import build as B

SLOTS = 4   # kAhead


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
def test_opening_requests_are_issued_slot_by_slot(tmp_path):
    out = str(tmp_path / "few.s")
    subprocess.run([B.HIPCC, *B.FLAGS, "--cuda-device-only", "-S", os.path.join(B.CSRC, "gemm_few.hip"), "-o", out], check=True,
                   stderr=subprocess.DEVNULL)
    kernels, loads, counted = {}, None, False
    for line in open(out):
        head = re.match(r"_ZN5ntfp815gemm_few_kernelILi\dELi\dELi(\d)ELi(\d)EEEv\w+:", line)
        if head:
            loads, counted = kernels.setdefault(line.split(":")[0], ((int(head[1]), int(head[2])), []))[1], False
        elif loads is not None and not counted:
            counted = "vmcnt" in line   # the first wait: everything before it is an opening request
            if re.match(r"\s+(buffer|global|flat)_load", line):
                loads.append(bool(re.search(r"\blds\b", line)))
    assert len(kernels) == 12
    for name, ((mi, nj), loads) in kernels.items():
        slot = 2 * nj + 2 * mi
        assert len(loads) == SLOTS * slot, name
        for s in range(SLOTS):
            assert sum(loads[s * slot:(s + 1) * slot]) == 2 * nj, (name, s)
