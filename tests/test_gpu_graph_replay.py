"""Calls captured into a HIP graph and replayed: a batched decode step (the sequential recurrence and a short attention call, which
hand data between workgroups) and short attention calls of every kind. Each replay has new input rows, follows an eager call, and is
compared bit for bit with the eager call on the same rows."""
import pytest

import hybrid_attention as ha
import synth
from harness import Runner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds,B,P,L", [
    (["linear_attention", "full_attention"], 8, 1536, 1), (["full_attention"], 1, 1531, 61), (["full_attention"], 3, 700, 40),
    (["full_attention"], 8, 0, 64), (["full_attention"], 1, 2900, 1)])
def test_replays_equal_eager_calls(kinds, B, P, L):
    import torch
    r = Runner(kinds, batch=B)
    st = torch.cuda.Stream()
    r.eng.set_stream(st.cuda_stream)
    rows, params = {"linear_attention": synth.gdn_rows, "full_attention": synth.gqa_rows}, {
        "linear_attention": synth.gdn_params(seed=41), "full_attention": synth.gqa_params(seed=41, noise=0.1)}
    for i, k in enumerate(kinds):
        r.set_params(i, params[k])
    _, snap = r.forward([rows[k](P, B, seed=42) for k in kinds], keep=True) if P else (None, None)
    steps = [[torch.from_numpy(rows[k](L, B, seed=43 + s)).to("cuda:0", dtype=r._dt(c)) for k, c in zip(kinds, r.kinds)]
             for s in range(4)]
    ins = [x.clone() for x in steps[0]]
    outs = [torch.empty(B, L, 2048, device="cuda:0", dtype=x.dtype) for x in ins]

    def call():
        r.eng.forward(L, ins, outs, cache=snap, recurrence=ha.SEQUENTIAL)

    def load(s):
        for a, b in zip(ins, steps[s]):
            a.copy_(b)
        for o in outs:
            o.fill_(float("nan"))

    torch.cuda.synchronize()
    want = []
    with torch.cuda.stream(st):
        for s in range(4):
            load(s)
            call()
            st.synchronize()
            want.append([o.clone() for o in outs])
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            call()
        for n, s in enumerate([1, 2, 2, 3, 0, 1, 3]):
            if n % 2:  # an eager call on other rows between two replays
                load((s + 1) % 4)
                call()
                st.synchronize()
            load(s)
            g.replay()
            st.synchronize()
            for o, w in zip(outs, want[s]):
                assert torch.equal(o, w), "replay %d" % n
    r.eng.synchronize()
