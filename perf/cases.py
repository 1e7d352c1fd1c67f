"""The work a user of libnnhip has it do, as cases that can be timed and
checked: one dict of plain values per case.

  listed()             the fixed cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  inputs, weights and handles a program holds beforehand
  run(state)           one pass through the public entry points
  work(case)           bytes and operations a pass cannot do without
  tolerance(case)      what another correct implementation may differ by
  exact(case, seed)    the same outputs in 64 bits, in plain torch

Kinds of case:

  linear_w8    one quantised Dense (QuantizedDense::forward): a projection of
               a decode step (a few rows), of a batched verify step (tens to
               hundreds) or of a prompt (thousands), INT8 or INT4 codes
  ln_linear    norm -> projection, the pair every decoder layer runs twice
  linear_f32   one Dense of a model that was not quantised
  attention    RoPE + KV append, then causal attention over the cache: the
               attention layer between its projections, for a decode or
               verify step (few new positions over many cached ones) or a
               prompt (all positions new), fp32 or int8 cache, grouped heads
  sample       get_probs + sample_token over the rows of a batch
  accept       the accept / resample step of speculative sampling
  mlp_train    the ExecutionBackend ops as a Tensor program calls them:
               forward and backward of a two-layer classifier
  generate     greedy speculative decoding of whole models, then the logits
               of what was generated (a program that reports token scores)
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "neural-network_amd", "python"))

import nnhip  # noqa: E402

DEV = "cuda"
F64 = torch.float64

# Decoder sizes of the two speculative-decoding configurations: a batch-1
# pair with a 4096-word vocabulary and a batch pair with 32000 words.
MODELS = {
    "small": dict(target=dict(V=4096, d=512, H=8, F=2048, L=6),
                  draft=dict(V=4096, d=256, H=4, F=1024, L=2)),
    "large": dict(target=dict(V=32000, d=1024, H=16, F=4096, L=12),
                  draft=dict(V=32000, d=512, H=8, F=2048, L=4)),
}
MAX_SEQ = 1024


def listed():
    return [
        # the gate/up projection of a batch-1 verify step (k + 1 = 5 rows)
        dict(name="linear_w8_decode", kind="linear_w8", rows=5, K=512, N=4096, bits=8),
        # the down projection of a batch-32 verify step (32 x 6 rows)
        dict(name="linear_w8_verify", kind="linear_w8", rows=192, K=4096, N=1024, bits=8),
        # norm + gate/up projection of a batch-32 prompt of 256 ids
        dict(name="ln_linear_prefill", kind="ln_linear", rows=8192, K=1024, N=8192),
        # a Dense of an unquantised model over a few prompts, odd sizes
        dict(name="linear_f32_prompt", kind="linear_f32", rows=333, K=772, N=1544),
        # the attention layer of a batch-32 verify step, fp32 cache
        dict(name="attention_verify", kind="attention", B=32, S=6, H=16, Hkv=16, D=64,
             cached=320, cap=1024, q8=False),
        # prompts through an attention layer with grouped query heads
        dict(name="attention_prompt", kind="attention", B=4, S=1000, H=16, Hkv=4, D=64,
             cached=0, cap=1024, q8=False),
        # a verify step over long contexts held in an int8 cache
        dict(name="attention_long_int8", kind="attention", B=16, S=8, H=8, Hkv=8, D=64,
             cached=2048, cap=2304, q8=True),
        # sampling a batch with top-k and top-p
        dict(name="sample_filtered", kind="sample", B=32, V=32000, T=0.8, top_k=50, top_p=0.9),
        # accept / resample of a large batch
        dict(name="accept_batch", kind="accept", B=256, k=8, V=32000, T=1.0),
        # a training step of a classifier on the backend's ops
        dict(name="mlp_train", kind="mlp_train", M=1024, I=784, H=1024, C=100),
        # batch-1 decoding
        dict(name="generate_b1", kind="generate", model="small", B=1, P=128, new=64, k=4,
             score=1, q8=False, bits=8),
        # batch decoding
        dict(name="generate_b32", kind="generate", model="large", B=32, P=256, new=64, k=5,
             score=4, q8=False, bits=8),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear_w8", "linear_w8", "ln_linear", "linear_f32", "attention",
                       "attention", "sample", "accept", "mlp_train", "generate"])
    if kind == "linear_w8":
        # model widths, and widths no tile divides (any multiple of 4)
        K = rng.choice([128, 256, 384, 512, 768, 1024, 1536, 2048, 3072, 4096,
                        4 * _log(rng, 16, 1024)])
        N = rng.choice([64 * _log(rng, 1, 128), _log(rng, 48, 8192)])
        return dict(kind=kind, rows=_log(rng, 1, 4096), K=K, N=N, bits=rng.choice([8, 8, 4]))
    if kind == "ln_linear":
        return dict(kind=kind, rows=_log(rng, 1, 8192), K=rng.choice([128, 256, 512, 1024]),
                    N=32 * _log(rng, 2, 256))
    if kind == "linear_f32":
        return dict(kind=kind, rows=_log(rng, 1, 2048),
                    K=rng.choice([128, 256, 512, 1024, 4 * _log(rng, 16, 1024)]),
                    N=_log(rng, 32, 8192))
    if kind == "attention":
        q8 = rng.random() < 0.4
        D = rng.choice([64, 64, 64, 32, 32, 16, 40])
        Hkv = rng.choice([2, 4, 8, 16] if D > 32 else [4, 8])
        H = Hkv if q8 else Hkv * rng.choice([1, 1, 2])
        prompt = rng.random() < 0.4
        S = _log(rng, 16, 1000) if prompt else rng.randint(1, 9)
        cached = rng.choice([0, 0, _log(rng, 1, 500)]) if prompt else _log(rng, 16, 2048)
        B = _log(rng, 1, 8 if prompt else 32)
        cap = cached + S + rng.choice([0, 17, 250])
        return dict(kind=kind, B=B, S=S, H=H, Hkv=Hkv, D=D, cached=cached, cap=cap, q8=q8)
    if kind == "sample":
        top_k, top_p = rng.choice([(0, 1.0), (50, 1.0), (0, 0.9), (40, 0.95)])
        return dict(kind=kind, B=_log(rng, 1, 256), V=_log(rng, 256, 32768),
                    T=rng.choice([0.0, 0.7, 1.0, 1.3]), top_k=top_k, top_p=top_p)
    if kind == "accept":
        return dict(kind=kind, B=_log(rng, 1, 256), k=rng.randint(1, 8),
                    V=_log(rng, 512, 32768), T=rng.choice([1.0, 0.8]))
    if kind == "mlp_train":
        return dict(kind=kind, M=_log(rng, 32, 2048), I=_log(rng, 32, 1024),
                    H=_log(rng, 32, 1024), C=_log(rng, 2, 1000))
    B = rng.choice([1, 1, 1, 2, 3, 8, 16])
    return dict(kind="generate", model="small", B=B, P=rng.randint(16, 300),
                new=rng.randint(16, 96), k=rng.randint(2, 7), score=1,
                q8=rng.random() < 0.3, bits=rng.choice([8, 8, 4]))


# ---------------------------------------------------------------- helpers ----
_CTX = None


def _ctx():
    """The program's one context."""
    global _CTX
    if _CTX is None:
        torch.cuda.init()
        _CTX = nnhip.Context(0)
    return _CTX


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _quantised(w, bits):
    """Codes [N][K] int8 and scales [N] of w [N][K]: symmetric, per output."""
    top = 127.0 if bits == 8 else 7.0
    s = w.abs().amax(1) / top
    s = torch.where(s == 0, torch.ones_like(s), s)
    return (w / s[:, None]).round().clamp(-top, top).to(torch.int8), s


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, device=DEV, dtype=dtype)


class _State(dict):
    """A program's handles; models and caches are freed with it."""

    def __del__(self):
        for h in self.get("handles", ()):
            h.free()


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return s


def run(state):
    return _RUN[state["case"]["kind"]](state)


def work(case):
    return _WORK[case["kind"]](case)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


# -------------------------------------------------- quantised projections ----
def _linear_inputs(case, seed):
    g = _gen(seed)
    K, N = case["K"], case["N"]
    # activations of a post-norm block: unit scale, a few outlying channels
    x = _randn(g, case["rows"], K)
    x[:, torch.randint(0, K, (max(1, K // 128),), generator=g, device=DEV)] *= 6.0
    w = _randn(g, N, K, std=0.02)
    return g, x, w, _randn(g, N, std=0.1)


def _prep_linear_w8(case, seed):
    _, x, w, bias = _linear_inputs(case, seed)
    codes, scales = _quantised(w, case["bits"])
    return _State(case=case, ctx=_ctx(), x=x, codes=codes.contiguous(), scales=scales,
                  bias=bias, y=_empty(case["rows"], case["N"]))


def _run_linear_w8(s):
    c = s["case"]
    nnhip.call("nnhip_linear_w8a32", s["ctx"].h, _p(s["x"]), c["rows"], c["K"], _p(s["codes"]),
               _p(s["scales"]), _p(s["bias"]), c["N"], _p(s["y"]), 0)
    return s["y"]


def _exact_linear_w8(case, seed):
    _, x, w, bias = _linear_inputs(case, seed)
    codes, scales = _quantised(w, case["bits"])
    return x.to(F64) @ (codes.to(F64) * scales.to(F64)[:, None]).T + bias.to(F64)


def _work_linear(case, code_bytes):
    r, K, N = case["rows"], case["K"], case["N"]
    return dict(bytes=4 * r * K + code_bytes * K * N + 8 * N + 4 * r * N, flops=2 * r * K * N)


# ----------------------------------------------------- norm -> projection ----
def _ln_inputs(case, seed):
    g, x, w, bias = _linear_inputs(case, seed)
    x = x + 0.3
    gamma = 1.0 + _randn(g, case["K"], std=0.1)
    return x, gamma, _randn(g, case["K"], std=0.1), w, bias


def _prep_ln_linear(case, seed):
    x, gamma, beta, w, bias = _ln_inputs(case, seed)
    codes, scales = _quantised(w, 8)
    return _State(case=case, ctx=_ctx(), x=x, gamma=gamma, beta=beta, codes=codes.contiguous(),
                  scales=scales, bias=bias, ln=_empty(case["rows"], case["K"]),
                  y=_empty(case["rows"], case["N"]))


def _run_ln_linear(s):
    c = s["case"]
    nnhip.call("nnhip_layernorm_linear_w8a32", s["ctx"].h, _p(s["x"]), c["rows"], c["K"],
               _p(s["gamma"]), _p(s["beta"]), _p(s["ln"]), _p(s["codes"]), _p(s["scales"]),
               _p(s["bias"]), c["N"], _p(s["y"]))
    return s["ln"], s["y"]


def _exact_ln_linear(case, seed):
    x, gamma, beta, w, bias = _ln_inputs(case, seed)
    codes, scales = _quantised(w, 8)
    x = x.to(F64)
    xc = x - x.mean(1, keepdim=True)
    ln = xc / (xc.square().mean(1, keepdim=True) + 1e-5).sqrt() * gamma.to(F64) + beta.to(F64)
    return ln, ln @ (codes.to(F64) * scales.to(F64)[:, None]).T + bias.to(F64)


def _work_ln_linear(case):
    w = _work_linear(case, 1)
    w["bytes"] += 4 * case["rows"] * case["K"] + 8 * case["K"]
    return w


# ------------------------------------------------------ fp32 projections ----
def _prep_linear_f32(case, seed):
    _, x, w, bias = _linear_inputs(case, seed)
    return _State(case=case, ctx=_ctx(), x=x, w=w, bias=bias, y=_empty(case["rows"], case["N"]))


def _run_linear_f32(s):
    c = s["case"]
    nnhip.call("nnhip_linear_f32", s["ctx"].h, _p(s["x"]), c["rows"], c["K"], _p(s["w"]),
               _p(s["bias"]), c["N"], _p(s["y"]))
    return s["y"]


def _exact_linear_f32(case, seed):
    _, x, w, bias = _linear_inputs(case, seed)
    return x.to(F64) @ w.to(F64).T + bias.to(F64)


# -------------------------------------------------------------- attention ----
def _attention_inputs(case, seed):
    g = _gen(seed)
    B, S, H, Hkv, D, cap = (case[n] for n in ("B", "S", "H", "Hkv", "D", "cap"))
    # ragged batch: sequence b has up to a quarter less than `cached` behind it
    lens = [max(0, case["cached"] - (b * 37 + seed * 11) % (case["cached"] // 4 + 1))
            for b in range(B)]
    qkv = _randn(g, B * S, (H + 2 * Hkv) * D)
    k = _randn(g, B, Hkv, cap, D)
    v = _randn(g, B, Hkv, cap, D)
    pos = torch.tensor(lens, dtype=torch.int32, device=DEV)
    return lens, pos, qkv, k, v


def _quantised_rows(x):
    """Codes and scales of rows along the last dimension (int8 KV rows)."""
    s = x.abs().amax(-1) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    y = x * (1.0 / s)[..., None]
    return (torch.sign(y) * (y.abs() + 0.5).floor()).clamp(-127, 127).to(torch.int8), s


def _prep_attention(case, seed):
    lens, pos, qkv, k, v = _attention_inputs(case, seed)
    s = _State(case=case, ctx=_ctx(), qkv=qkv, pos=pos,
               q=_empty(case["B"] * case["S"], case["H"] * case["D"]),
               out=_empty(case["B"] * case["S"], case["H"] * case["D"]))
    if case["q8"]:
        s["k"], s["ks"] = _quantised_rows(k)
        s["v"], s["vs"] = _quantised_rows(v)
    else:
        s["k"], s["v"] = k, v
    return s


def _run_attention(s):
    c, h = s["case"], s["ctx"].h
    B, S, H, Hkv, D, cap = (c[n] for n in ("B", "S", "H", "Hkv", "D", "cap"))
    if c["q8"]:
        nnhip.call("nnhip_rope_kv_append_q8", h, _p(s["qkv"]), B, S, H, D, _p(s["pos"]), _p(s["q"]),
                   _p(s["k"]), _p(s["ks"]), _p(s["v"]), _p(s["vs"]), cap)
        nnhip.call("nnhip_attention_kq_q8", h, _p(s["q"]), _p(s["k"]), _p(s["ks"]), _p(s["v"]),
                   _p(s["vs"]), cap, _p(s["pos"]), B, S, H, Hkv, D, _p(s["out"]))
        return s["out"], s["k"], s["ks"], s["v"], s["vs"]
    nnhip.call("nnhip_rope_kv_append_gqa", h, _p(s["qkv"]), B, S, H, Hkv, D, _p(s["pos"]),
               _p(s["q"]), _p(s["k"]), _p(s["v"]), cap)
    nnhip.call("nnhip_attention_kq", h, _p(s["q"]), _p(s["k"]), _p(s["v"]), cap, _p(s["pos"]),
               B, S, H, Hkv, D, _p(s["out"]))
    return s["out"], s["k"], s["v"]


def _rope64(x, start, D):
    """x [heads][S][D] rotated at positions start + s: the angles are the
    float32 ones the format prescribes, their cosines and the products are
    formed in 64 bits."""
    theta = np.power(10000.0, -2.0 * np.arange(D // 2, dtype=np.float32) / np.float32(D),
                     dtype=np.float64).astype(np.float32)
    w = (np.arange(start, start + x.shape[1], dtype=np.float32)[:, None] * theta).astype(np.float64)
    c, s = (torch.from_numpy(f(w)).to(x.device) for f in (np.cos, np.sin))
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack((e * c - o * s, e * s + o * c), -1).flatten(-2)


def _attend64(q, k, v, past):
    """Causal attention of q [H][S][D] over k, v [Hkv][past + S][D]."""
    H, S, D = q.shape
    k, v = (t.repeat_interleave(H // t.shape[0], 0) for t in (k, v))
    out = torch.empty_like(q)
    for h in range(H):
        sc = q[h] @ k[h].T / math.sqrt(D)
        mask = torch.ones(S, past + S, dtype=torch.bool, device=q.device).triu(past + 1)
        out[h] = torch.softmax(sc.masked_fill(mask, -math.inf), -1) @ v[h]
    return out


def _exact_attention(case, seed):
    B, S, H, Hkv, D = (case[n] for n in ("B", "S", "H", "Hkv", "D"))
    lens, _, qkv, k, v = _attention_inputs(case, seed)
    q8 = case["q8"]
    if q8:
        (kc, ks), (vc, vs) = _quantised_rows(k), _quantised_rows(v)
    k, v = k.to(F64), v.to(F64)
    out = torch.empty(B, S, H * D, device=DEV, dtype=F64)
    rows = qkv.to(F64).view(B, S, H + 2 * Hkv, D).transpose(1, 2)
    for b, n in enumerate(lens):
        q = _rope64(rows[b, :H], n, D)
        k[b, :, n:n + S] = _rope64(rows[b, H:H + Hkv], n, D)
        v[b, :, n:n + S] = rows[b, H + Hkv:]
        kb, vb = k[b, :, :n + S], v[b, :, :n + S]
        if q8:
            sl = slice(n, n + S)
            kc[b, :, sl], ks[b, :, sl] = _quantised_rows(k[b, :, sl].float())
            vc[b, :, sl], vs[b, :, sl] = _quantised_rows(v[b, :, sl].float())
            kb = kc[b, :, :n + S].to(F64) * ks[b, :, :n + S].to(F64)[..., None]
            vb = vc[b, :, :n + S].to(F64) * vs[b, :, :n + S].to(F64)[..., None]
        out[b] = _attend64(q, kb, vb, n).transpose(0, 1).reshape(S, H * D)
    out = out.view(B * S, H * D)
    return (out, kc, ks.to(F64), vc, vs.to(F64)) if q8 else (out, k, v)


def _work_attention(case):
    B, S, H, Hkv, D = (case[n] for n in ("B", "S", "H", "Hkv", "D"))
    keys = sum(max(0, case["cached"] - (b * 37) % (case["cached"] // 4 + 1)) for b in range(B))
    row = D + 4 if case["q8"] else 4 * D
    pairs = S * keys + B * S * (S + 1) // 2           # (query, visible key)
    return dict(bytes=B * S * (H + 2 * Hkv) * D * 4 + 2 * Hkv * row * (keys + B * S)
                + B * S * H * D * 4, flops=4 * D * H * pairs)


# ---------------------------------------------------------------- sampling ----
def _sample_inputs(case, seed):
    g = _gen(seed)
    logits = _randn(g, case["B"], case["V"], std=2.5)
    return logits, torch.rand(case["B"], generator=g, device=DEV)


def _prep_sample(case, seed):
    logits, u = _sample_inputs(case, seed)
    B, V = case["B"], case["V"]
    return _State(case=case, ctx=_ctx(), logits=logits, u=u, tok=_empty(B, dtype=torch.int32),
                  probs=_empty(B, V) if case["T"] > 0 else None)


def _run_sample(s):
    c = s["case"]
    nnhip.call("nnhip_sample_rows", s["ctx"].h, _p(s["logits"]), c["B"], c["V"], c["T"],
               c["top_k"], c["top_p"], _p(s["u"]), _p(s["tok"]),
               _p(s["probs"]) if c["T"] > 0 else None)
    return (s["tok"], s["probs"]) if c["T"] > 0 else (s["tok"],)


def _invert64(w, u):
    """First index whose running sum of w reaches u * sum(w), per row."""
    cs = w.cumsum(-1)
    at = (cs < u.to(F64)[:, None] * cs[:, -1:]).sum(-1)
    return at.clamp(max=w.shape[-1] - 1).to(torch.int32)


def _exact_sample(case, seed):
    logits, u = _sample_inputs(case, seed)
    if case["T"] <= 0:
        return (logits.argmax(-1).to(torch.int32),)
    V = case["V"]
    p = torch.softmax(logits.to(F64) / float(np.float32(case["T"])), -1)
    order = torch.sort(p, dim=-1, descending=True, stable=True)
    keep = torch.ones_like(p, dtype=torch.bool)
    if 0 < case["top_k"] < V:
        keep[:, case["top_k"]:] = False
    if 0 < case["top_p"] < 1:
        cs = (order.values * keep).cumsum(-1)
        keep[:, 1:] &= cs[:, :-1] < float(np.float32(case["top_p"]))
    p = torch.where(torch.zeros_like(keep).scatter(-1, order.indices, keep), p, torch.zeros_like(p))
    p = p / p.sum(-1, keepdim=True)
    return _invert64(p, u), p


def _accept_inputs(case, seed):
    g = _gen(seed)
    B, k, V = case["B"], case["k"], case["V"]
    # a draft that follows its target: about three of four drafts accepted
    d = _randn(g, B, k, V, std=2.0)
    t = d + _randn(g, B, k, V, std=0.7)
    noise = torch.empty_like(d).exponential_(generator=g)
    tok = (torch.softmax(d / case["T"], -1) / noise).argmax(-1).to(torch.int32)
    ua = torch.rand(B, k, generator=g, device=DEV)
    return t, d, tok, ua, torch.rand(B, generator=g, device=DEV)


def _prep_accept(case, seed):
    t, d, tok, ua, ur = _accept_inputs(case, seed)
    B = case["B"]
    return _State(case=case, ctx=_ctx(), t=t, d=d, tok=tok, ua=ua, ur=ur,
                  n=_empty(B, dtype=torch.int32), next=_empty(B, dtype=torch.int32))


def _run_accept(s):
    c = s["case"]
    nnhip.call("nnhip_spec_accept", s["ctx"].h, _p(s["t"]), _p(s["d"]), _p(s["tok"]), _p(s["ua"]),
               _p(s["ur"]), c["B"], c["k"], c["V"], c["T"], _p(s["n"]), _p(s["next"]))
    return s["n"], s["next"]


def _exact_accept(case, seed):
    t, d, tok, ua, ur = _accept_inputs(case, seed)
    k, T = case["k"], float(np.float32(case["T"]))
    n = torch.zeros(case["B"], dtype=torch.int64, device=DEV)
    nxt = torch.full((case["B"],), -1, dtype=torch.int32, device=DEV)
    live = torch.ones(case["B"], dtype=torch.bool, device=DEV)
    for j in range(k):
        p, q = (torch.softmax(x[:, j].to(F64) / T, -1) for x in (t, d))
        c = tok[:, j:j + 1].long()
        ok = ua[:, j].to(F64) * q.gather(1, c)[:, 0] < p.gather(1, c)[:, 0]
        draw_ = _invert64((p - q).clamp(min=0), ur)
        nxt = torch.where(live & ~ok, draw_, nxt)
        live = live & ok
        n += live
    return n.to(torch.int32), nxt


# ------------------------------------------------------ backend training ----
def _mlp_inputs(case, seed):
    g = _gen(seed)
    M, I, H, C = case["M"], case["I"], case["H"], case["C"]
    x = torch.rand(M, I, generator=g, device=DEV)
    y = torch.nn.functional.one_hot(torch.randint(0, C, (M,), generator=g, device=DEV), C).float()
    return (x, y, _randn(g, I, H, std=math.sqrt(2.0 / I)), _randn(g, H, std=0.05),
            _randn(g, H, C, std=math.sqrt(2.0 / H)), _randn(g, C, std=0.05))


def _view(t, shape=None, strides=None):
    v = nnhip.View()
    v.data = t.data_ptr()
    shape = tuple(t.shape) if shape is None else shape
    strides = tuple(t.stride()) if strides is None else strides
    v.offset, v.rank = 0, len(shape)
    for i, (n, st) in enumerate(zip(shape, strides)):
        v.shape[i], v.strides[i] = n, st
    return v


def _prep_mlp(case, seed):
    x, y, w1, b1, w2, b2 = _mlp_inputs(case, seed)
    M, I, H, C = case["M"], case["I"], case["H"], case["C"]
    t = dict(x=x, y=y, w1=w1, b1=b1, w2=w2, b2=b2,
             inv=torch.full((1,), 1.0 / M, device=DEV))
    for n, shape in dict(a1=(M, H), z1=(M, H), h=(M, H), a2=(M, C), z2=(M, C), p=(M, C),
                         e=(M, C), g=(M, C), dh=(M, H), dz=(M, H), dw1=(I, H), db1=(H,),
                         dw2=(H, C), db2=(C,)).items():
        t[n] = _empty(*shape)
    v = {n: _view(a) for n, a in t.items()}
    for n in ("x", "h", "w2"):                        # transposed views
        a = t[n]
        v[n + "T"] = _view(a, (a.shape[1], a.shape[0]), (a.stride(1), a.stride(0)))
    return _State(case=case, ctx=_ctx(), t=t, v={n: ctypes.byref(a) for n, a in v.items()},
                  keep=v, axis0=(ctypes.c_int64 * 1)(0))


def _run_mlp(s):
    h, v, t = s["ctx"].h, s["v"], s["t"]

    def mm(a, b, o):
        nnhip.call("nnhip_matmul_f32", h, v[a], v[b], v[o])

    def binary(op, a, b, o):
        nnhip.call("nnhip_binary_f32", h, op, v[a], v[b], v[o])

    mm("x", "w1", "a1")
    binary(nnhip.OP_ADD, "a1", "b1", "z1")
    nnhip.call("nnhip_unary_f32", h, nnhip.OP_RELU, v["z1"], v["h"])
    mm("h", "w2", "a2")
    binary(nnhip.OP_ADD, "a2", "b2", "z2")
    nnhip.call("nnhip_softmax_f32", h, v["z2"], v["p"], 1)
    # cross entropy: d z2 = (p - y) / M
    binary(nnhip.OP_SUB, "p", "y", "e")
    binary(nnhip.OP_MUL, "e", "inv", "g")
    mm("hT", "g", "dw2")
    nnhip.call("nnhip_sum_f32", h, v["g"], v["db2"], s["axis0"], 1)
    mm("g", "w2T", "dh")
    binary(nnhip.OP_RELU_BACKWARD, "z1", "dh", "dz")
    mm("xT", "dz", "dw1")
    nnhip.call("nnhip_sum_f32", h, v["dz"], v["db1"], s["axis0"], 1)
    return {n: t[n] for n in ("p", "dw1", "db1", "dw2", "db2")}


def _exact_mlp(case, seed):
    x, y, w1, b1, w2, b2 = (a.to(F64) for a in _mlp_inputs(case, seed))
    z1 = x @ w1 + b1
    h = z1.clamp(min=0)
    p = torch.softmax(h @ w2 + b2, -1)
    g = (p - y) / case["M"]
    dz = (g @ w2.T) * (z1 > 0)
    return dict(p=p, dw1=x.T @ dz, db1=dz.sum(0), dw2=h.T @ g, db2=g.sum(0))


def _work_mlp(case):
    M, I, H, C = case["M"], case["I"], case["H"], case["C"]
    return dict(bytes=4 * (M * I + 2 * M * C + 2 * (I * H + H + H * C + C)),
                flops=4 * M * I * H + 6 * M * H * C)


# -------------------------------------------------------------- generation ----
def _decoder_params(cfg, nxt, g):
    """Parameters (TransformerDecoder::parameters() order) of a decoder whose
    most likely next token after v is nxt[v]: N(0, 0.02) layers, as a fresh
    model has them, and an lm head aligned with the embedding of the
    predecessor, so that the logits are as peaked as a trained model's."""
    V, d, F, L = cfg["V"], cfg["d"], cfg["F"], cfg["L"]
    emb = _randn(g, V, d)
    p = [emb]
    zero, one = torch.zeros(d, device=DEV), torch.ones(d, device=DEV)
    for _ in range(L):
        for _ in range(4):
            p += [_randn(g, d, d, std=0.02), zero]
        p += [_randn(g, d, F, std=0.02), torch.zeros(F, device=DEV)]
        p += [_randn(g, d, F, std=0.02), torch.zeros(F, device=DEV)]
        p += [_randn(g, F, d, std=0.02), zero]
        p += [one, zero, one, zero]
    head = _randn(g, d, V, std=0.02)
    head.index_add_(1, nxt, emb.T / math.sqrt(d))
    return p + [head, torch.zeros(V, device=DEV)]


def _generate_inputs(case, seed):
    g = _gen(seed)
    m = MODELS[case["model"]]
    V = m["target"]["V"]
    nxt = torch.randperm(V, generator=g, device=DEV)
    # the draft agrees with the target on four of five tokens
    other = torch.randint(0, V, (V,), generator=g, device=DEV)
    dn = torch.where(torch.rand(V, generator=g, device=DEV) < 0.8, nxt, other)
    prompts = torch.randint(0, V, (case["B"], case["P"]), generator=g, device=DEV)
    return m, prompts, _decoder_params(m["target"], nxt, g), lambda: _decoder_params(m["draft"], dn, g)


def _prep_generate(case, seed):
    m, prompts, tp, draft = _generate_inputs(case, seed)
    s = _State(case=case, ctx=_ctx(), handles=[])
    for name, params in (("target", tp), ("draft", draft())):
        c = m[name]
        mod = nnhip.Decoder(s["ctx"], c["V"], c["d"], c["H"], c["F"], c["L"], MAX_SEQ)
        s["handles"].insert(0, mod)
        mod.set_params([a.cpu().numpy() for a in params])
        mod.quantize(case["bits"])
        s[name] = mod
    s["prompts"] = prompts.cpu().numpy().astype(np.int32)
    # the scored sequences' prompts are already in a cache of the target
    n = case["score"]
    s["cache"] = nnhip.KVCache(s["target"], n)
    s["handles"].insert(0, s["cache"])
    s["target"].forward(s["prompts"][:n, :-1], s["cache"])
    return s


def _run_generate(s):
    c = s["case"]
    out, _, _ = s["target"].generate_speculative_batch(
        s["draft"], s["prompts"], c["new"], c["k"], 0.0, 42, quantized_cache=c["q8"])
    n, P = c["score"], c["P"]
    logits = s["target"].forward(out[:n, P - 1:-1], s["cache"])
    for b in range(n):
        s["cache"].truncate(P - 1, b)
    return out, logits


def _forward64(p, cfg, ids, past):
    """Logits of ids [B][S] after the cached k, v of `past` (updated)."""
    H, L = cfg["H"], cfg["L"]
    D = cfg["d"] // H
    B, S = ids.shape
    x = p[0][ids]

    def norm(h, g, b):
        c = h - h.mean(-1, keepdim=True)
        return c / (c.square().mean(-1, keepdim=True) + 1e-5).sqrt() * g + b

    for i in range(L):
        (wq, bq, wk, bk, wv, bv, wo, bo, wg, bg, wu, bu, wd, bd, g1, b1, g2, b2) = p[1 + 18 * i:19 + 18 * i]
        q, k, v = ((x @ w + b).view(B, S, H, D).transpose(1, 2) for w, b in ((wq, bq), (wk, bk), (wv, bv)))
        n = past[i][0].shape[2] if past[i] else 0
        q, k = (_rope64(t.reshape(B * H, S, D), n, D).view(B, H, S, D) for t in (q, k))
        if past[i]:
            k, v = torch.cat((past[i][0], k), 2), torch.cat((past[i][1], v), 2)
        past[i] = (k, v)
        sc = q @ k.transpose(2, 3) / math.sqrt(D)
        mask = torch.ones(S, n + S, dtype=torch.bool, device=x.device).triu(n + 1)
        a = torch.softmax(sc.masked_fill(mask, -math.inf), -1) @ v
        x = norm(x + a.transpose(1, 2).reshape(B, S, H * D) @ wo + bo, g1, b1)
        x = norm(x + (torch.nn.functional.silu(x @ wg + bg) * (x @ wu + bu)) @ wd + bd, g2, b2)
    return x @ p[-2] + p[-1]


def _exact_generate(case, seed):
    m, prompts, params, _ = _generate_inputs(case, seed)
    cfg = m["target"]
    p = []
    for i, a in enumerate(params):
        # the Dense weights [in][out] are quantised per output, the rest is not
        dense = i == len(params) - 2 or (0 < i < len(params) - 2 and (i - 1) % 18 < 14 and (i - 1) % 2 == 0)
        if dense:
            codes, s = _quantised(a.T.contiguous(), case["bits"])
            a = (codes.to(F64) * s.to(F64)[:, None]).T
        p.append(a.to(F64))
    past = [None] * cfg["L"]
    # greedy speculative decoding gives the target's own greedy tokens
    B, n = case["B"], case["score"]
    x = _forward64(p, cfg, prompts[:, :-1], past)[:, :0]
    toks, logits, last = [prompts], [], prompts[:, -1:]
    for _ in range(case["new"]):
        x = _forward64(p, cfg, last, past)
        logits.append(x[:n])
        last = x.argmax(-1)
        toks.append(last)
    return torch.cat(toks, 1).to(torch.int32), torch.cat(logits, 1)


def _work_generate(case):
    m = MODELS[case["model"]]
    B, P, new, k = (case[n] for n in ("B", "P", "new", "k"))

    def dense(c):
        return c["L"] * (4 * c["d"] * c["d"] + 3 * c["d"] * c["F"])

    def kv(c, keys):
        return c["L"] * 2 * keys * (c["d"] + 4 * c["H"] if case["q8"] else 4 * c["d"])

    t, d = m["target"], m["draft"]
    head = {id(c): c["d"] * c["V"] for c in (t, d)}
    # at the 0.8 agreement a cycle commits 1 + sum_j 0.8^j tokens
    per = 1 + sum(0.8 ** j for j in range(1, k + 1))
    cycles = max(1, math.ceil((new - 1) / per))
    mid = P + new // 2
    bts = (dense(t) + dense(d) + head[id(t)]                              # prefill
           + cycles * (dense(t) + head[id(t)] + B * kv(t, mid))           # verify
           + cycles * k * (dense(d) + head[id(d)] + B * kv(d, mid)))      # drafting
    flops = 2 * (B * P * (dense(t) + dense(d))
                 + cycles * B * (k + 1) * (dense(t) + head[id(t)])
                 + cycles * B * k * (dense(d) + head[id(d)]))
    scored = case["score"] * new
    bts += dense(t) + head[id(t)] + case["score"] * kv(t, mid) + 4 * scored * t["V"]
    flops += 2 * scored * (dense(t) + head[id(t)])
    return dict(bytes=bts, flops=flops)


_PREPARE = dict(linear_w8=_prep_linear_w8, ln_linear=_prep_ln_linear, linear_f32=_prep_linear_f32,
                attention=_prep_attention, sample=_prep_sample, accept=_prep_accept,
                mlp_train=_prep_mlp, generate=_prep_generate)
_RUN = dict(linear_w8=_run_linear_w8, ln_linear=_run_ln_linear, linear_f32=_run_linear_f32,
            attention=_run_attention, sample=_run_sample, accept=_run_accept, mlp_train=_run_mlp,
            generate=_run_generate)
_EXACT = dict(linear_w8=_exact_linear_w8, ln_linear=_exact_ln_linear, linear_f32=_exact_linear_f32,
              attention=_exact_attention, sample=_exact_sample, accept=_exact_accept,
              mlp_train=_exact_mlp, generate=_exact_generate)
_WORK = dict(
    linear_w8=lambda c: _work_linear(c, 1 if c["bits"] == 8 else 0.5),
    ln_linear=_work_ln_linear,
    linear_f32=lambda c: _work_linear(c, 4),
    attention=_work_attention,
    sample=lambda c: dict(bytes=4 * c["B"] * c["V"] * (2 if c["T"] > 0 else 1) + 8 * c["B"], flops=0),
    # rows up to the first rejection, about 0.75 accepted each
    accept=lambda c: dict(bytes=8 * c["B"] * c["V"] * sum(0.75 ** j for j in range(c["k"])), flops=0),
    mlp_train=_work_mlp,
    generate=_work_generate,
)


def tolerance(case):
    return _TOLERANCE[case["kind"]]


# About four times the relative errors against exact() that were measured:
# the digit planes of a quantised Dense resolve 2^-22 of a row's maximum, the
# fp32 sums of the others about 1e-7; in generate that travels through the
# layers.  differ: int8 cache codes and drawn tokens at a rounding boundary.
_TOLERANCE = dict(
    linear_w8=dict(rel=5e-6),
    ln_linear=dict(rel=5e-6),
    linear_f32=dict(rel=1e-6),
    attention=dict(rel=1e-6, differ=1e-4),
    sample=dict(rel=2e-6, differ=0.01),
    accept=dict(differ=0.01),
    mlp_train=dict(rel=3e-6),
    generate=dict(rel=3e-4),
)
