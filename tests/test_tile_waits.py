"""Guard on the compiled gfx950 code of mnb_tiles_kernel: a wave's part of an LDS copy has landed before the barrier that hands
the tile to the other waves. The copies are written out (lds_dma.h), so the compiler does not wait for them by itself, and a wave
whose columns all lie past N executes no other wait. The check follows every path of a kernel's control flow with the vector memory
operations it may have in flight (they complete in order; s_waitcnt vmcnt(n) leaves the last n) and asks that at each s_barrier at
most one tile's copies are: the ones for the tile after next. Kernels of every format and tile shape."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"
CSRC = os.path.join(ROOT, "strands-decider-web_amd", "csrc")

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is missing")


def blocks_of(lines):
    """Basic blocks {label: ([operation], [successor])}; operations: "dma", "vm", "barrier" or the count n of a vmcnt(n)."""
    blocks, name = {}, "entry"
    ops, nxt, open_ = [], [], True

    def close(fall):
        blocks[name] = (ops, nxt + ([fall] if fall and open_ else []))

    n = 0
    for l in lines:
        m = re.match(r"^(\.L\w+):", l)
        if m:
            close(m.group(1))
            name, ops, nxt, open_ = m.group(1), [], [], True
            continue
        l = l.split(";")[0].strip()
        if not l or l.startswith("."):
            continue
        op = l.split()[0]
        if op.startswith("global_load_lds"):
            ops.append("dma")
        elif op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            ops.append("vm")
        elif op == "s_barrier":
            ops.append("barrier")
        elif op == "s_waitcnt":
            c = re.search(r"vmcnt\((\d+)\)", l)
            assert c or "lgkmcnt" in l or "expcnt" in l, "a wait written as a number: " + l
            if c:
                ops.append(int(c.group(1)))
        elif op == "s_endpgm":
            open_ = False
        elif op.startswith(("s_cbranch", "s_branch")):
            nxt.append(l.split()[1])
            n += 1
            if op == "s_branch":
                open_ = False
            close("+%d" % n)
            name, ops, nxt, open_ = "+%d" % n, [], [], True
    close(None)
    return blocks


def copies_at_barriers(blocks):
    """The largest number of copies that some path has in flight at a barrier."""
    seen, todo, worst, barriers = set(), [("entry", ())], 0, 0
    while todo:
        at = todo.pop()
        if at in seen:
            continue
        seen.add(at)
        assert len(seen) < 500000, "too many states"
        name, flight = at
        ops, nxt = blocks[name]
        for op in ops:
            if op == "barrier":
                worst, barriers = max(worst, sum(flight)), barriers + 1
            elif isinstance(op, int):
                flight = flight[-op:] if op else ()
            else:
                flight = (flight + (op == "dma",))[-63:]
        todo += [(x, flight) for x in nxt]
    return worst, barriers


def test_the_check_finds_a_missing_wait():
    code = ["global_load_lds_dwordx4 v1, s[0:1]", "global_load_dwordx4 v[2:5], v[0:1], off", ".L1:",
            "global_load_lds_dwordx4 v1, s[0:1]", "s_cbranch_scc1 .L2", "s_waitcnt vmcnt(1)", ".L2:", "s_barrier",
            "s_cbranch_scc0 .L1", "s_endpgm"]
    assert copies_at_barriers(blocks_of(code))[0] > 1
    code[4] = "s_nop 0"
    assert copies_at_barriers(blocks_of(code))[0] == 1


def test_copies_have_landed_at_every_barrier(tmp_path):
    out = tmp_path / "mnb.s"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-x", "hip", "-S",
                        "--cuda-device-only", os.path.join(CSRC, "mnb.hip"), "-o", str(out)],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    bad, kernels = [], 0
    for m in re.finditer(r"^(_Z\w*mnb_tiles_kernel\w*):.*?^\.Lfunc_end", out.read_text(), re.M | re.S):
        group, asym, rt, ct, wm, wn = (int(x) for x in re.search(r"kernelI" + r"L[ib](\d+)E" * 6, m.group(1)).groups())
        copies = 32 * rt * wm // 8 // (wm * wn)  # copy instructions of a wave for one tile, 8 rows each
        worst, barriers = copies_at_barriers(blocks_of(m.group(0).splitlines()[1:]))
        assert barriers
        kernels += 1
        if worst > copies:
            bad.append((group, asym, rt, ct, wm, wn, "copies in flight at a barrier: %d, one tile is %d" % (worst, copies)))
    assert kernels == 12
    assert not bad, bad
