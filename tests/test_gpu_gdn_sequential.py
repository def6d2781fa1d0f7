"""GPU parity of the sequential gated-delta kernel (decode / resume path) against the fp64 oracle."""
import numpy as np
import pytest

import hybrid_attention as ha
import synth
from harness import Runner, gdn_inputs, oracle_gdn, rel_err

pytestmark = pytest.mark.gpu
TOL = 2e-3  # north-star bar for the fp32 recurrence (max |err| / max |ref|)


def _state(snap, B=1):
    s = np.zeros((B, 16, 128, 128), np.float32)
    return snap.read(0, "state", s)


@pytest.mark.parametrize("gnorm", [False, True])
def test_config0_sequential(gnorm):
    # the CPU-runnable case: T=64, 16 heads, fp32 rows, conv taps N(0, 0.5^2), negA = -1, dt_bias = 0, S0 = 0
    x = gdn_inputs(64)
    p = synth.gdn_params()
    r = Runner(["linear_attention"], gnorm=gnorm)
    r.set_params(0, p)
    (out,), snap = r.forward([x], keep=True, recurrence=ha.SEQUENTIAL)
    ref, st = oracle_gdn(x, p, gnorm=gnorm)
    e = rel_err(out, ref)
    print("config0 sequential gnorm=%s rel_err out %.2e" % (gnorm, e))
    assert e < TOL
    es = rel_err(_state(snap)[0], st[0].S)
    print("state rel_err %.2e" % es)
    assert es < TOL
    assert snap.P == 64 and snap.state_pos == 64 and snap.tail_rows == 3


def test_sequential_batch_f16_rows():
    B, T = 3, 50
    x = gdn_inputs(T, B, seed=1, dtype=np.float16)
    p = synth.gdn_params(seed=1, neg_exp_A=-0.3, dt_bias=0.5)
    r = Runner(["linear_attention"], batch=B, lin_dtype=ha.F16)
    r.set_params(0, p)
    (out,), _ = r.forward([x], recurrence=ha.SEQUENTIAL)
    ref, _ = oracle_gdn(x.astype(np.float32), p)
    e = rel_err(out, ref)
    print("B=3 f16 rows rel_err %.2e" % e)
    assert e < 1e-2  # f16 output rounding (2^-11) plus the fp32 recurrence


@pytest.mark.parametrize("P,L", [(37, 27), (1, 5), (64, 64), (3, 1)])
def test_sequential_prefix_suffix_bit_exact(P, L):
    x = gdn_inputs(P + L, 2, seed=2)
    p = synth.gdn_params(seed=2)
    r = Runner(["linear_attention"], batch=2)
    r.set_params(0, p)
    (full,), fsnap = r.forward([x], keep=True, recurrence=ha.SEQUENTIAL)
    (pre,), snap = r.forward([x[:, :P]], keep=True, recurrence=ha.SEQUENTIAL)
    (suf,), ssnap = r.forward([x[:, P:]], cache=snap, keep=True, recurrence=ha.SEQUENTIAL)
    np.testing.assert_array_equal(pre, full[:, :P])
    np.testing.assert_array_equal(suf, full[:, P:])
    np.testing.assert_array_equal(_state(ssnap, 2), _state(fsnap, 2))


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("T", [1, 2, 63, 66, 131])
def test_many_sequences_equal_few(T, f16):
    # launches of more than 512 workgroups (9 sequences of 16 heads) load the gated norm's factors after the last token: the
    # same rows as in an engine of 3 sequences, and for one of them the oracle's
    B, dt = 9, np.float16 if f16 else np.float32
    x, p = gdn_inputs(T, B, seed=4, dtype=dt), synth.gdn_params(seed=4)
    many, few = (Runner(["linear_attention"], batch=b, lin_dtype=ha.F16 if f16 else ha.F32) for b in (B, 3))
    for r in (many, few):
        r.set_params(0, p)
    (out,), _ = many.forward([x], recurrence=ha.SEQUENTIAL)
    for b in range(0, B, 3):
        (o,), _ = few.forward([x[b:b + 3]], recurrence=ha.SEQUENTIAL)
        if f16:  # (a product's last rounding, f32 first or not, is the compiler's choice: one unit of an f16 result)
            np.testing.assert_allclose(out[b:b + 3], o, rtol=2 ** -10, atol=1e-7)
        else:
            np.testing.assert_array_equal(out[b:b + 3], o)
    ref, _ = oracle_gdn(x[8:9].astype(np.float32), p)
    assert rel_err(out[8:9], ref) < (1e-2 if f16 else TOL)
