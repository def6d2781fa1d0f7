"""Short full-attention calls (gqa_rows.h) at the edges of their groups, tiles and pieces: every row equals, bit for bit,
the same row of one long forward, which runs the general kernel; rows of both types; the caches a short call writes; a
wait that runs out is reported."""
import numpy as np
import pytest

import hybrid_attention as ha
import synth
from harness import Runner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("B,P,steps", [
    (1, 0, [1, 31, 32, 33]), (1, 63, [1, 1, 64, 65, 256]), (1, 509, [3, 129, 255]), (1, 1983, [64, 1]),
    (2, 0, [128, 1]), (3, 191, [1, 33, 96, 128]), (8, 60, [5, 64]), (16, 100, [32, 64, 7]),
    (2, 2030, [17, 1, 33, 128]), (3, 2900, [1, 100])])
def test_rows_equal_a_long_forward(B, P, steps, f32):
    # the long forward has more rows than any short call: the general kernel; contexts of more than 2048 positions have more
    # tiles than the values kernel holds in LDS at a time
    T = max(P + sum(steps), 300)
    x = synth.gqa_rows(T, B, seed=31)
    x = x.astype(np.float32) if f32 else x
    r = Runner(["full_attention"], batch=B, max_ctx=2048 if T <= 2048 else 4096, **({"full_dtype": ha.F32} if f32 else {}))
    r.set_params(0, synth.gqa_params(seed=31, noise=0.1))
    (full,), whole = r.forward([x], keep=True)
    s, a = None, P
    if P:
        (_,), s = r.forward([x[:, :P]], keep=True)
    for L in steps:
        (o,), s = r.forward([x[:, a:a + L]], cache=s, keep=True)
        np.testing.assert_array_equal(o, full[:, a:a + L], err_msg="rows %d..%d" % (a, a + L))
        a += L
    for part in ("K", "V"):
        got, want = np.zeros((B, 2, a, 256), np.float16), np.zeros((B, 2, T, 256), np.float16)
        s.read(0, part, got)
        whole.read(0, part, want)
        np.testing.assert_array_equal(got, want[:, :, :a], err_msg=part)


@pytest.mark.parametrize("stride,off", [(5124, 0), (5120, 4), (5132, 4)])
def test_rows_that_are_not_16_byte_aligned(stride, off):
    # a row stride or a first row at a multiple of 8 bytes only: the same bits as 16-byte aligned rows
    import torch
    x = torch.from_numpy(synth.gqa_rows(300, 1, seed=33)).to("cuda:0")
    outs = []
    for st, of in ((5120, 0), (stride, off)):
        e = ha.Engine(ha.model_config(["full_attention"], batch=1, max_ctx=512, full_stride=st))
        for n, v in synth.gqa_params(seed=33, noise=0.1).items():
            e.set_param(0, n, v)
        buf = torch.zeros(300 * st + of + 8, dtype=torch.float16, device="cuda:0")
        rows = buf[of:of + 300 * st].view(300, st)
        rows[:, :5120] = x[0]
        o = torch.empty(1, 300, 2048, dtype=torch.float16, device="cuda:0")
        torch.cuda.synchronize()
        snap = e.forward(200, [rows], [o], keep_cache=True, sync=True)["cache"]
        for a, b in ((200, 261), (200, 209)):
            o2 = torch.empty(1, b - a, 2048, dtype=torch.float16, device="cuda:0")
            torch.cuda.synchronize()
            e.forward(b - a, [rows[a:]], [o2], cache=snap, sync=True)
            outs.append((st, of, o2))
        outs.append((st, of, o[:, :200].clone()))
    for (_, _, w), (_, _, g) in zip(outs[:3], outs[3:]):
        assert torch.equal(w, g)


def test_wait_that_runs_out_is_reported():
    import torch
    x = torch.from_numpy(synth.gqa_rows(200, 1, seed=32)).to("cuda:0")
    o = torch.empty(1, 200, 2048, dtype=torch.float16, device="cuda:0")
    r = Runner(["full_attention"], batch=1, max_ctx=512)
    r.set_params(0, synth.gqa_params(seed=32))
    torch.cuda.synchronize()
    r.eng.forward(200, [x], [o], sync=True)
    want = o.clone()
    with pytest.raises(ha.HAError) as ei:
        r.eng.forward(200, [x], [o], sync=True, debug_unpublished_waits=True)
    assert ei.value.code == ha.HA_ERR_DEVICE and "gave up waiting" in str(ei.value)
    r.eng.forward(200, [x], [o], sync=True)
    assert torch.equal(o, want)
