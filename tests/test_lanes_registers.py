"""Guard on the compiled gfx950 code of the one- and two-row projections: their block and scale arrays are in registers. (As arrays
of 16-bit values the compiler had put the scales in scratch memory, or in LDS at odd addresses, four times the kernel's time.)"""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"
CSRC = os.path.join(ROOT, "strands-decider-web_amd", "csrc")

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is missing")


def test_no_array_is_kept_in_memory(tmp_path):
    out = tmp_path / "mnb.s"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-x", "hip", "-S",
                        "--cuda-device-only", os.path.join(CSRC, "mnb.hip"), "-o", str(out)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    seen, bad = 0, []
    for m in re.finditer(r"^\s+\.amdhsa_kernel (\S*mnb_gemv_(?:lanes|wide)_kernel\S*)(.*?)\.end_amdhsa_kernel", out.read_text(), re.M | re.S):
        seen += 1
        for what in ("group_segment_fixed_size", "private_segment_fixed_size"):  # (the staged rows of a are dynamic LDS)
            n = int(re.search(what + r"\s+(\d+)", m.group(2)).group(1))
            if n:
                bad.append((m.group(1), what, n))
    assert seen == 48  # 12 formats, one or two rows, two or four columns a wave
    assert not bad, bad
