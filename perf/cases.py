"""The calls whose speed this framework is judged by: what a host program has it do, through its public entry points.

Five kinds of call, at the shapes of the model the framework is built for (hidden size 2048, MLP width 6144, 16
gated-delta heads of 128, 8 query and 2 KV heads of 256, int4 weights in blocks of 32):

  gdn    one gated-delta layer over the fused in_proj rows: prefill, a suffix resumed from a prefix snapshot, decode
  gqa    one full-attention layer over the fused qkv rows: prefill, a resumed suffix, decode
  mnb    one quantised projection y = a W^T
  mlp    one MLP block: residual add + norm, (rotation,) gate_up, SiLU gate, (rotation,) down
  torso  a whole forward, embedding to final norm, of the model's 16 layers

A host keeps the engine, the weights and the prefix snapshot between calls, so these belong to the prepared state; the
rows, activations and token ids of a call are its inputs."""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "strands-decider-web_amd"))
import hybrid_attention as ha  # noqa: E402

DEV = "cuda:0"
D, I, VOCAB = 2048, 6144, 4096
H, DK, LIN_STRIDE, LIN_W = 16, 128, 8256, 8224          # in_proj rows: q k v (6144) | z (2048) | a b (32) | padding
HQ, HK, HD, RD, FULL_STRIDE = 8, 2, 256, 64, 5120       # qkv rows: [q | gate] x 8 | k x 2 | v x 2
MAX_CTX, THETA, EPS = 4096, 1e7, 1e-6
# (N, K) of the projections: gate_up, down, in_proj, qkv, out_proj / o_proj / adapter
SHAPES = [(2 * I, D), (D, I), (8256, D), (5120, D), (D, D)]
# 11 gated-delta, 4 full-attention and 1 adapter layer: the counts of the model's matmuls per forward
LAYERS = (["linear_attention"] * 3 + ["full_attention"]) * 3 + ["linear_attention"] * 2 + ["adapter", "full_attention"]


def listed():
    return [
        # the headline prefill's gated-delta layer: eight sequences of 2048 tokens, fp32 rows
        dict(name="gdn prefill 8x2048 f32", kind="gdn", B=8, P=0, L=2048, f16=False, recurrence="chunked"),
        # the layer of a torso forward that prefills one state document of odd length
        dict(name="gdn prefill 1x1531 f16", kind="gdn", B=1, P=0, L=1531, f16=True, recurrence="chunked"),
        # a question resumed from the cached state
        dict(name="gdn resume 1x1531+61 f16", kind="gdn", B=1, P=1531, L=61, f16=True, recurrence="chunked"),
        # one decode step of a batch
        dict(name="gdn decode 8x1536+1 f32", kind="gdn", B=8, P=1536, L=1, f16=False, recurrence="sequential"),
        # the headline prefill's attention layer
        dict(name="gqa prefill 8x2048 f16", kind="gqa", B=8, P=0, L=2048, f16=True),
        # a question's attention over the cached state
        dict(name="gqa resume 1x1531+61 f16", kind="gqa", B=1, P=1531, L=61, f16=True),
        # one decode step of a batch
        dict(name="gqa decode 8x1536+1 f16", kind="gqa", B=8, P=1536, L=1, f16=True),
        # a decode step's largest projection (weight bandwidth)
        dict(name="mnb gate_up M=1", kind="mnb", M=1, N=2 * I, K=D, bits=4, group=32, asym=False),
        # a short question's projections, the long reduction
        dict(name="mnb down M=61", kind="mnb", M=61, N=D, K=I, bits=4, group=32, asym=False),
        # a long prefill's input projection
        dict(name="mnb in_proj M=2048", kind="mnb", M=2048, N=8256, K=D, bits=4, group=32, asym=False),
        # an MLP block whose weights were exported with the input rotation
        dict(name="mlp M=333 rotated", kind="mlp", M=333, had=True),
        # a whole question on a cached state, the call of a decision
        dict(name="torso 1531+68", kind="torso", P=1531, L=68),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gdn", "gdn", "gqa", "gqa", "mnb", "mnb", "mnb", "mlp", "torso"])
    if kind == "mnb":
        N, K = rng.choice(SHAPES)
        bits, group, asym = rng.choice([(4, 32, False)] * 4 + [(4, 64, False), (4, 32, True), (3, 32, False), (2, 64, True)])
        if rng.random() < 0.25:  # another model's widths
            N, K = 16 * _spread(rng, 16, 512), 64 * _spread(rng, 8, 96)
        return dict(kind=kind, M=_spread(rng, 1, 2048), N=N, K=K, bits=bits, group=group, asym=asym)
    if kind == "mlp":
        return dict(kind=kind, M=_spread(rng, 1, 1024), had=rng.random() < 0.5)
    if kind == "torso":
        return dict(kind=kind, P=rng.choice([0, _spread(rng, 32, 2048)]), L=_spread(rng, 4, 68))
    B = rng.choice([1, 1, 1, 2, 3, 4, 5, 8])
    P = _spread(rng, 16, 2040) if rng.random() < 0.6 else 0
    L = _spread(rng, 1, 128 if P else 2047)
    case = dict(kind=kind, B=B, P=P, L=L, f16=rng.random() < (0.5 if kind == "gdn" else 0.8))
    if kind == "gdn":
        case["recurrence"] = "sequential" if P and L <= 8 else "chunked"
    return case


# ---- inputs ----

_stream = None


def _one_stream():
    """The stream that every engine of the program runs on: its calls follow one another."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream

def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + stream)


def _rows(kind, B, T, f16, g):
    """Rows as a projection of normalised activations leaves them: ~N(0, 1), the stride's padding zero."""
    w, stride = (LIN_W, LIN_STRIDE) if kind == "gdn" else (FULL_STRIDE, FULL_STRIDE)
    x = torch.zeros(B, T, stride, device=DEV, dtype=torch.float16 if f16 else torch.float32)
    for b in range(B):
        x[b, :, :w] = torch.randn(T, w, device=DEV, generator=g)
    return x


def _mixer_params(kind, rng):
    f = np.float32
    if kind == "gdn":
        return {"conv": (0.5 * rng.standard_normal((3 * H * DK, 4))).astype(f),
                "neg_exp_A": (-np.exp(rng.uniform(-2.0, 1.0, H))).astype(f),
                "dt_bias": (0.5 * rng.standard_normal(H)).astype(f),
                "gnorm": (1 + 0.1 * rng.standard_normal(DK)).astype(f)}
    return {n: (1 + 0.1 * rng.standard_normal(HD)).astype(f) for n in ("q_norm", "k_norm")}


def _weight(N, K, bits, group, asym, g):
    """Packed blocks of a roughly normal, zero-mean matrix of random codes, with f16 scales (and biases)."""
    mid = 2 ** (bits - 1)
    c = torch.randn(N, K // 32, 32, device=DEV, generator=g).mul_(mid / 3).add_(mid).round_().clamp_(0, 2 * mid - 1).int()
    if bits == 4:
        q = torch.stack([sum(c[..., 8 * j + i] << (4 * i) for i in range(8)) for j in range(4)], -1)
    else:
        q = torch.stack([sum((c[..., 16 * j + i] & 3) << (2 * i) for i in range(16)) for j in range(2)], -1)
        if bits == 3:
            q = torch.cat([q, sum((c[..., i] >> 2) << i for i in range(32))[..., None]], -1)
    s = ((0.03 + 0.01 * torch.rand(N, K // group, device=DEV, generator=g)) / mid).to(torch.float16)
    b = (-mid * s.float() + 0.004 * torch.randn(N, K // group, device=DEV, generator=g)).to(torch.float16) if asym else None
    return {"N": N, "K": K, "bits": bits, "group": group, "asym": asym, "q": q.int().contiguous(), "s": s, "b": b}


def _handle(w):
    return ha.MnbWeight(w["N"], w["K"], w["q"], w["s"], w["b"], bits=w["bits"], group=w["group"], asym=w["asym"])


def _mixer_data(case, seed):
    g = _gen(seed, 1)
    return {"params": _mixer_params(case["kind"], np.random.default_rng([int(seed), 2])),
            "prefix": _rows(case["kind"], case["B"], case["P"], case["f16"], g) if case["P"] else None,
            "rows": _rows(case["kind"], case["B"], case["L"], case["f16"], g)}


def _mnb_data(case, seed):
    g = _gen(seed, 3)
    return {"w": _weight(case["N"], case["K"], case["bits"], case["group"], case["asym"], g),
            "a": torch.randn(case["M"], case["K"], device=DEV, generator=g).to(torch.float16)}


def _mlp_data(case, seed):
    g, M = _gen(seed, 4), case["M"]
    return {"x": torch.randn(M, D, device=DEV, generator=g),
            "y": (0.3 * torch.randn(M, D, device=DEV, generator=g)).to(torch.float16),
            "norm": 1 + 0.1 * torch.randn(D, device=DEV, generator=g),
            "gate_up": _weight(2 * I, D, 4, 32, False, g), "down": _weight(D, I, 4, 32, False, g)}


def _torso_data(case, seed):
    g, rng = _gen(seed, 5), np.random.default_rng([int(seed), 6])
    vec = lambda: (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)  # noqa: E731
    W, V, X = {"embed": _weight(VOCAB, D, 4, 32, False, g)}, {"final_norm": vec()}, {}
    for i, t in enumerate(LAYERS):
        p = "layers.%d." % i
        V[p + "in_norm"] = vec()
        if t == "adapter":
            W[p + "proj"] = _weight(D, D, 4, 32, False, g)
            V[p + "bias"] = (0.05 * rng.standard_normal(D)).astype(np.float32)
            continue
        lin = t == "linear_attention"
        W[p + ("in_proj" if lin else "qkv")] = _weight(8256 if lin else 5120, D, 4, 32, False, g)
        W[p + ("out_proj" if lin else "o_proj")] = _weight(D, D, 4, 32, False, g)
        V[p + "post_norm"] = vec()
        W[p + "gate_up"] = _weight(2 * I, D, 4, 32, False, g)
        W[p + "down"] = _weight(D, I, 4, 32, False, g)
        X[i] = _mixer_params("gdn" if lin else "gqa", rng)
    return {"W": W, "V": V, "X": X, "prefix": rng.integers(0, VOCAB, case["P"]).tolist(),
            "ids": rng.integers(0, VOCAB, case["L"]).tolist()}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("gdn", "gqa"):
        d = _mixer_data(case, seed)
        B, L = case["B"], case["L"]
        dt, code = (torch.float16, ha.F16) if case["f16"] else (torch.float32, ha.F32)
        layer = "linear_attention" if kind == "gdn" else "full_attention"
        e = ha.Engine(ha.model_config([layer], batch=B, max_ctx=MAX_CTX, lin_dtype=code, full_dtype=code),
                      stream=_one_stream().cuda_stream)
        for n, v in d["params"].items():
            e.set_param(0, n, v)
        s = {"kind": kind, "engine": e, "L": L, "rows": d["rows"],
             "out": torch.empty(B, L, D, device=DEV, dtype=dt), "cache": None,
             "mode": ha.SEQUENTIAL if case.get("recurrence") == "sequential" else ha.CHUNKED}
        torch.cuda.synchronize()
        if case["P"]:
            o = torch.empty(B, case["P"], D, device=DEV, dtype=dt)
            s["cache"] = e.forward(case["P"], [d["prefix"]], [o], keep_cache=True)["cache"]
            torch.cuda.synchronize()
        return s
    if kind == "mnb":
        d = _mnb_data(case, seed)
        return {"kind": kind, "w": _handle(d["w"]), "M": case["M"], "a": d["a"],
                "y": torch.empty(case["M"], case["N"], device=DEV, dtype=torch.float16)}
    if kind == "mlp":
        d, M = _mlp_data(case, seed), case["M"]
        f16 = torch.float16
        return {"kind": kind, "M": M, "had": case["had"], "x": d["x"], "y": d["y"], "norm": d["norm"],
                "gate_up": _handle(d["gate_up"]), "down": _handle(d["down"]),
                "h": torch.empty(M, D, device=DEV, dtype=f16), "big": torch.empty(M, 2 * I, device=DEV, dtype=f16),
                "mid": torch.empty(M, I, device=DEV, dtype=f16), "out": torch.empty(M, D, device=DEV, dtype=f16)}
    d = _torso_data(case, seed)
    t = ha.Torso(LAYERS, D=D, I=I, max_ctx=MAX_CTX)
    for n, w in d["W"].items():
        t.set_weight(n, _handle(w))
    for n, v in d["V"].items():
        t.set_param(n, v)
    for i, params in d["X"].items():
        for n, v in params.items():
            t.set_param("layers.%d.%s" % (i, n), v)
    cache = t.forward(d["prefix"], [], keep=True)[1] if case["P"] else None
    torch.cuda.synchronize()
    return {"kind": kind, "torso": t, "ids": d["ids"], "cache": cache}


# ---- one pass ----

def run(s):
    kind = s["kind"]
    if kind in ("gdn", "gqa"):
        s["engine"].forward(s["L"], [s["rows"]], [s["out"]], cache=s["cache"],
                            **({"recurrence": s["mode"]} if kind == "gdn" else {}))
        return s["out"]
    if kind == "mnb":
        s["w"].forward(s["M"], s["a"], s["y"])
        return s["y"]
    if kind == "mlp":
        M = s["M"]
        ha.add_norm(M, D, M, s["x"], s["y"], s["norm"], s["h"])
        if s["had"]:
            ha.fwht(s["h"], M * D, D)
        s["gate_up"].forward(M, s["h"], s["big"])
        ha.silu_mul(M, I, s["big"], s["mid"])
        if s["had"]:
            ha.fwht(s["mid"], M * I, D)
        s["down"].forward(M, s["mid"], s["out"])
        return {"x": s["x"], "out": s["out"]}
    return s["torso"].forward(s["ids"], cache=s["cache"])[0]


# ---- what a pass cannot do without ----

def _mnb_bytes(N, K, bits=4, group=32, asym=False):
    return N * K * bits // 8 + N * (K // group) * 2 * (2 if asym else 1)


def work(case):
    kind = case["kind"]
    if kind == "gdn":
        B, L, e = case["B"], case["L"], 2 if case["f16"] else 4
        # rows in, rows out, the state read where there is one; per token and head 3 products with the 128 x 128 state
        return {"bytes": B * L * (LIN_W + D) * e + (B * H * DK * DK * 4 if case["P"] else 0),
                "flops": B * L * H * 3 * 2 * DK * DK}
    if kind == "gqa":
        B, L, P, e = case["B"], case["L"], case["P"], 2 if case["f16"] else 4
        return {"bytes": B * L * (FULL_STRIDE + D) * e + B * P * 2 * HK * HD * 2,
                "flops": B * 4 * HQ * HD * (L * (L + 1) // 2 + P * L)}
    if kind == "mnb":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _mnb_bytes(N, K, case["bits"], case["group"], case["asym"]) + 2 * M * (N + K), "flops": 2 * M * N * K}
    if kind == "mlp":
        M = case["M"]
        return {"bytes": _mnb_bytes(2 * I, D) + _mnb_bytes(D, I) + M * D * (4 + 4 + 2 + 2), "flops": 2 * M * 3 * I * D}
    P, L = case["P"], case["L"]
    lin, full = LAYERS.count("linear_attention"), LAYERS.count("full_attention")
    per_token = lin * (8256 * D + D * D) + full * (5120 * D + D * D) + (lin + full) * 3 * I * D + D * D
    return {"bytes": per_token * 9 // 16 + lin * H * DK * DK * 4 * (1 if P else 0) + full * (P + L) * 2 * HK * HD * 2 + L * D * 4,
            "flops": 2 * L * per_token + full * 4 * HQ * HD * (L * (L + 1) // 2 + P * L) + lin * L * H * 3 * 2 * DK * DK}


def tolerance(case):
    # About four times the path's measured distance from its 64-bit value (f16 operands, weights or rows and fp32 sums:
    # gdn 2.2e-4..4.8e-4, gqa 3.7e-4..4.3e-4, mnb 2.8e-4, mlp 7e-4; the torso's 16 layers carry it to 8e-3).
    return {"rel": {"gdn": 1.8e-3, "gqa": 1.7e-3, "mnb": 1.1e-3, "mlp": 2.8e-3, "torso": 3e-2}[case["kind"]],
            "max": {"gdn": 2e-2, "gqa": 2e-2, "mnb": 6e-3, "mlp": 2e-2, "torso": 0.2}[case["kind"]]}


# ---- the same in 64 bits ----

def _silu(x):
    return x * torch.sigmoid(x)


def _gdn64(rows, p, skip):
    """The sequential gated-delta rule over rows [B][T][stride], with conv, norms, gates and gated norm; rows skip.. out."""
    p = {k: torch.from_numpy(v).double().to(DEV) for k, v in p.items()}
    B, T = rows.shape[:2]
    C = 3 * H * DK
    S = torch.zeros(B, H, DK, DK, dtype=torch.float64, device=DEV)
    out = torch.empty(B, T - skip, H * DK, dtype=torch.float64, device=DEV)
    hist = torch.zeros(B, 3, C, dtype=torch.float64, device=DEV)
    for t0 in range(0, T, 256):  # blocks of rows: the f64 copies stay small
        r = rows[:, t0:t0 + 256].double()
        n = r.shape[1]
        x = torch.cat([hist, r[..., :C]], 1)
        hist = x[:, -3:]
        u = _silu(sum(x[:, j:j + n] * p["conv"][:, j] for j in range(4))).reshape(B, n, 3, H, DK)
        q, k, v = u[:, :, 0], u[:, :, 1], u[:, :, 2]
        q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + EPS) / math.sqrt(DK)
        k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + EPS)
        z = r[..., C:C + H * DK].reshape(B, n, H, DK)
        a, b = r[..., C + H * DK:C + H * DK + H], r[..., C + H * DK + H:C + H * DK + 2 * H]
        beta = torch.sigmoid(b)
        alpha = torch.exp(p["neg_exp_A"] * torch.nn.functional.softplus(a + p["dt_bias"]))
        for t in range(n):
            S *= alpha[:, t, :, None, None]
            d = (v[:, t] - (S * k[:, t, :, :, None]).sum(2)) * beta[:, t, :, None]
            S += k[:, t, :, :, None] * d[:, :, None, :]
            if t0 + t >= skip:
                o = (S * q[:, t, :, :, None]).sum(2)
                o = p["gnorm"] * o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS) * _silu(z[:, t])
                out[:, t0 + t - skip] = o.reshape(B, -1)
    return out


def _gqa64(rows, p, skip):
    """Causal attention over rows [B][T][stride] with q/k norms, partial RoPE and output gate; rows skip.. out."""
    p = {k: torch.from_numpy(v).double().to(DEV) for k, v in p.items()}
    B, T = rows.shape[:2]
    ang = torch.arange(T, dtype=torch.float64, device=DEV)[:, None] * \
        THETA ** (-torch.arange(0, RD, 2, dtype=torch.float64, device=DEV) / RD)
    cos, sin = ang.cos(), ang.sin()

    def prep(x, w):
        x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w
        x1, x2 = x[..., :RD // 2], x[..., RD // 2:RD]
        return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin, x[..., RD:]], -1)

    out = torch.empty(B, T - skip, HQ * HD, dtype=torch.float64, device=DEV)
    mask = torch.arange(T, device=DEV)[None, :] > torch.arange(skip, T, device=DEV)[:, None]
    for b in range(B):
        r = rows[b].double()
        for h in range(HQ):
            kh = HQ * 2 * HD + (h // (HQ // HK)) * HD
            q = prep(r[:, h * 2 * HD:h * 2 * HD + HD], p["q_norm"])[skip:]
            s = (q @ prep(r[:, kh:kh + HD], p["k_norm"]).T.contiguous()) / math.sqrt(HD)
            o = torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ r[:, kh + HK * HD:kh + HK * HD + HD]
            out[b, :, h * HD:(h + 1) * HD] = o * torch.sigmoid(r[skip:, h * 2 * HD + HD:(h + 1) * 2 * HD])
    return out


def _dequant64(w):
    """Codes of the packed blocks (4 bits: nibble e % 8 of word e / 8; 2 bits: bits 2 (e % 16) of word e / 16; 3 bits:
    the same low bits and bit e of word 2 above them), times the scale, as stored in f16."""
    q, bits = w["q"].long() & 0xFFFFFFFF, w["bits"]
    e = torch.arange(32, device=DEV)
    if bits == 4:
        c = (q[..., e // 8] >> (4 * (e % 8))) & 15
    else:
        c = (q[..., e // 16] >> (2 * (e % 16))) & 3
        if bits == 3:
            c = c | (((q[..., 2:3] >> e) & 1) << 2)
    c = c.reshape(w["N"], -1, w["group"]).double()
    s = w["s"].double()[..., None]
    c = c * s + w["b"].double()[..., None] if w["asym"] else (c - 2 ** (bits - 1)) * s
    return c.reshape(w["N"], w["K"])


def _mm64(a, w):
    return a @ _dequant64(w).T.contiguous()


def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rotate64(x, n):
    """The orthonormal Walsh-Hadamard transform (Sylvester order) of each n-block."""
    shape, h = x.shape, 1
    while h < n:
        x = x.reshape(-1, 2, h)
        x = torch.stack([x[:, 0] + x[:, 1], x[:, 0] - x[:, 1]], 1)
        h *= 2
    return x.reshape(shape) / math.sqrt(n)


def _mlp64(h, gate_up, down, had):
    big = _mm64(_rotate64(h, D) if had else h, gate_up)
    mid = _silu(big[:, :I]) * big[:, I:]
    return _mm64(_rotate64(mid, D) if had else mid, down)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gdn", "gqa"):
        d = _mixer_data(case, seed)
        rows = d["rows"] if d["prefix"] is None else torch.cat([d["prefix"], d["rows"]], 1)
        return (_gdn64 if kind == "gdn" else _gqa64)(rows, d["params"], case["P"])
    if kind == "mnb":
        d = _mnb_data(case, seed)
        return _mm64(d["a"].double(), d["w"])
    if kind == "mlp":
        d = _mlp_data(case, seed)
        x = d["x"].double() + d["y"].double()
        return {"x": x, "out": _mlp64(_norm64(x, d["norm"]), d["gate_up"], d["down"], case["had"])}
    d = _torso_data(case, seed)
    V = {n: torch.from_numpy(v).to(DEV) for n, v in d["V"].items()}
    W = d["W"]
    x, y = _dequant64(W["embed"])[torch.tensor(d["prefix"] + d["ids"], device=DEV)], 0
    for i, t in enumerate(LAYERS):
        p = "layers.%d." % i
        x = x + y
        h = _norm64(x, V[p + "in_norm"])
        if t == "adapter":
            y = _mm64(h, W[p + "proj"]) + V[p + "bias"].double()
            continue
        if t == "linear_attention":
            o = _mm64(_gdn64(_mm64(h, W[p + "in_proj"])[None], d["X"][i], 0)[0], W[p + "out_proj"])
        else:
            o = _mm64(_gqa64(_mm64(h, W[p + "qkv"])[None], d["X"][i], 0)[0], W[p + "o_proj"])
        x = x + o
        y = _mlp64(_norm64(x, V[p + "post_norm"]), W[p + "gate_up"], W[p + "down"], False)
    return _norm64((x + y)[case["P"]:], V["final_norm"])
