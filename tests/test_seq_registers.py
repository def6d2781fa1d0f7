"""Guard on the compiled gfx950 code of the sequential gated-delta kernel: the form for many sequences leaves room for four
workgroups a CU (128 registers a wave), which is what it is for."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"
CSRC = os.path.join(ROOT, "strands-decider-web_amd", "csrc")

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is missing")


def test_many_sequences_leave_room_for_four_workgroups(tmp_path):
    out = tmp_path / "seq.s"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-x", "hip", "-S",
                        "--cuda-device-only", os.path.join(CSRC, "gdn_seq.hip"), "-o", str(out)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    regs = {}
    for m in re.finditer(r"^\s+\.amdhsa_kernel \S*gdn_seq_kernelI(\w+?)Lb(\d)\S*(.*?)\.end_amdhsa_kernel", out.read_text(), re.M | re.S):
        regs[m.group(1), int(m.group(2))] = int(re.search(r"next_free_vgpr\s+(\d+)", m.group(3)).group(1))
    assert len(regs) == 4, regs
    for (_, early), n in regs.items():
        assert n <= (256 if early else 128), regs
