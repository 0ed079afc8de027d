"""The FP6 conversions (v_cvt_scalef32_2xpk16_fp6_f32, v_cvt_scalef32_pk32_f32_fp6) write their first
results before they have read their last operands, which the compiler does not know: a build
whose register allocation places the one over the other computes wrong terms.  The library's own
assembly, compiled with the flags of the build, must hold no such instruction."""
import os
import re
import shutil
import subprocess

import pytest

from __graft_entry__ import HIPCC_FLAGS, ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def _registers(operand):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]|v(\d+)", operand.strip())
    if not m:
        return set()
    lo, hi = (m[1], m[2]) if m[1] else (m[3], m[3])
    return set(range(int(lo), int(hi) + 1))


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_no_conversion_writes_over_its_operands(tmp_path):
    src, out = os.path.join(ROOT, "coalsack_amd", "csrc"), str(tmp_path / "capi.s")
    flags = [f for f in HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([HIPCC, *flags, "-S", "--cuda-device-only", "-I" + src, "-I" + os.path.join(ROOT, "include"),
                    os.path.join(src, "capi.hip"), "-o", out], check=True, capture_output=True, timeout=600)
    n = 0
    with open(out) as f:
        for line in f:
            m = re.match(r"\s*v_cvt_scalef32_(?:2xpk16_fp6_f32|pk32_f32_fp6)\s+([^;]*)", line)
            if m:
                result, *operands = (_registers(o) for o in m[1].split(", "))
                assert result and operands and not any(result & o for o in operands), line
                n += 1
    assert n > 100  # every kernel that quantises has three of one and two of the other per block
