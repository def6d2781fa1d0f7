"""Guard on the compiled gfx950 code of the full-attention kernels: the rotated q pairs are rounded by the one instruction written out
in gqa_common.h, in the general and in the short-call kernels. (Left to the compiler, which of a pair's two products is fused
depended on the rest of the kernel, and the two kernels' rows then differed in a bit here and there.)"""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"
CSRC = os.path.join(ROOT, "strands-decider-web_amd", "csrc")

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is missing")


def test_rotated_pairs_are_rounded_by_the_written_instruction(tmp_path):
    out = tmp_path / "gqa.s"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-x", "hip", "-S",
                        "--cuda-device-only", os.path.join(CSRC, "gqa.hip"), "-o", str(out)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    seen = 0
    for m in re.finditer(r"^(_Z\w*gqa_(?:attn|scores)_kernel\w*):.*?^\.Lfunc_end", out.read_text(), re.M | re.S):
        seen += 1
        code = m.group(0)
        mine = re.findall(r";;#ASMSTART\s+(v_fma_mixlo_f16)", code)
        assert len(mine) == 32, (m.group(1), len(mine))  # dims 0 .. 63: 16 pairs of 2 k-steps, two results each
        # (the f32 kernels' and the sums of squares' own forms give f32)
        assert len(re.findall(r"v_fma_mix(?:lo|hi)_f16", code)) == 32, m.group(1)
    assert seen == 8
