"""Raw-row tails of many gated-delta layers. The engine gathers the tail copies of one call into launches of up to
32 layers, or launches one per layer when per-layer times are asked for. With 35 gated-delta layers, both launch
forms (32 + 3 layers, and 35 single ones) must leave tails that resume bit-exactly. A suffix resumed from a prefix
snapshot must equal the same rows of one longer forward, for every layer (resume engine.js:325-328; conv history
roll wgsl.js:420-434). The prefix (100 rows) ends inside a chunk, so every tail holds replay rows as well as the
conv history."""
import numpy as np
import pytest

import hybrid_attention as ha
import synth
from harness import Runner

pytestmark = pytest.mark.gpu
N = 35


def _inputs(T, part, B):
    return [synth.gdn_rows(T, B, seed=5, layer=i, part=part) for i in range(N)]


@pytest.mark.parametrize("batch,layer_ms", [(1, False), (3, False), (3, True)])
def test_many_layer_tails_resume_bit_exact(batch, layer_ms):
    print("tails: %d gated-delta layers, batch %d, layer_ms %s" % (N, batch, layer_ms), flush=True)
    r = Runner(["linear_attention"] * N, batch=batch)
    for i in range(N):
        r.set_params(i, synth.gdn_params(seed=5, layer=i))
    prefix, suffix = _inputs(100, 0, batch), _inputs(37, 1, batch)
    _, snap = r.forward(prefix, keep=True, layer_ms=layer_ms)
    assert snap.P == 100 and snap.state_pos == 64
    outs, _ = r.forward(suffix, cache=snap, layer_ms=layer_ms)
    full, _ = r.forward([np.concatenate([p, q], 1) for p, q in zip(prefix, suffix)], layer_ms=layer_ms)
    for i in range(N):
        assert np.isfinite(outs[i]).all(), i
        np.testing.assert_array_equal(outs[i], full[i][:, 100:], err_msg="layer %d" % i)
    snap.release()


@pytest.mark.parametrize("f16", [False, True])
def test_tail_reads_the_rows_and_zeros(f16):
    # the raw rows of a snapshot as a host reads them: conv channels, a and b as they came in, the other columns zero, and the
    # same bytes in a block whose place of the rows held an earlier snapshot's K and V (three raw rows, then 1920 positions)
    B, C, AB = 2, 6144, 8192
    dt = np.float16 if f16 else np.float32
    r = Runner(["linear_attention", "full_attention"], batch=B, lin_dtype=ha.F16 if f16 else ha.F32)
    r.set_params(0, synth.gdn_params(seed=6))
    x = [synth.gdn_rows(180, B, seed=6).astype(dt), synth.gqa_rows(180, B, seed=6)]
    for n in range(2):
        _, snap = r.forward(x, keep=True)
        assert (snap.state_pos, snap.tail_rows) == (128, 55)
        g = snap.read(0, "tail", np.full((B, 55, 8256), 3, dt))
        np.testing.assert_array_equal(g[..., :C], x[0][:, 125:, :C])
        np.testing.assert_array_equal(g[..., AB:AB + 32], x[0][:, 125:, AB:AB + 32])
        assert not g[..., C:AB].any() and not g[..., AB + 32:].any(), n
        if n == 0:  # a larger block, which the next snapshot takes (the engine keeps one released block)
            _, large = r.forward([synth.gdn_rows(1920, B, seed=7).astype(dt), synth.gqa_rows(1920, B, seed=7)], keep=True)
            large.release()
