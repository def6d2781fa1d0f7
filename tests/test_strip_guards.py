"""Guard on the compiled gfx950 code of the files whose LDS DMAs are written out (lds_dma.h): a DMA sets m0, a register the compiler reserves and does not
preserve across asm, right before the instruction. Sound only while every m0 reference is the asm's own set."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is missing")


@pytest.mark.parametrize("name,kernels", [("torso.hip", "mnb_strip_kernel"), ("gqa.hip", "gqa_rows")])
def test_m0_is_written_only_by_the_dma_asm(tmp_path, name, kernels):
    out = tmp_path / "out.s"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"),
                        "-I" + os.path.join(ROOT, "strands-decider-web_amd", "csrc"), "-x", "hip", "-S",
                        "--cuda-device-only", os.path.join(ROOT, "strands-decider-web_amd", "csrc", name),
                        "-o", str(out)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    seen = 0
    for m in re.finditer(r"^(_Z\w*%s\w*):.*?^\.Lfunc_end" % kernels, out.read_text(), re.M | re.S):
        code = [l for l in (l.strip() for l in m.group(0).splitlines()) if l and not l.startswith((";", "."))]
        refs = [i for i, l in enumerate(code) if re.search(r"\bm0\b", l)]
        seen += len(refs)
        for i in refs:
            assert code[i].startswith("s_mov_b32 m0,"), (m.group(1), code[i])
            assert code[i + 1].startswith("global_load_lds_dword"), (m.group(1), code[i], code[i + 1])
    assert seen
