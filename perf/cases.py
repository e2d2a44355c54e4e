"""The work that programs on this framework have it do, as cases that can be timed.

A case is one pass of one of five kinds through the public entry points (the C
ABI of include/atlas_kernels.h on device buffers, and OlmoModel):

  mlp    the feed-forward block of one layer over `rows` activation rows: fused
         gate/up + SwiGLU, the down projection, the post-norm RMSNorm.  One row
         is decode, 2..16 rows a ragged batch's step, more a chunk of a prompt.
  attn   the attention block of one layer for one new token: residual + RMSNorm
         and QKV projection, QK-norm, RoPE, cache write and attention over `ctx`
         positions, output projection.  By the one-launch entry point
         ("fused") or by the three that a program keeping the reference's
         kernel boundary calls ("steps").
  head   the end of a token: final norm and lm_head, then its choice (greedy,
         or one of the two sampling presets).
  quant  encoding of a weight matrix when a checkpoint is loaded.
  model  a whole model: a prompt is fed, then `steps` tokens one by one, whose
         logits come back.

Weights are N(0, 0.02) stored as bf16, int8 (a scale per row) or int4 (a scale
per block of the flattened matrix); activations are normal with a log-normal
scale per channel, as a residual stream has.
"""
import ctypes as C
import math

import numpy as np
import torch

from atlas_amd import _lib
from atlas_amd import model as am

FMT = {"bf16": 1, "int8": 2, "int4": 3}
DEV = "cuda"
EPS = 1e-6


def listed():
    return [
        # one decode step's feed-forward of a 135M-sized model: the smallest call, all latency
        dict(name="mlp_135m_int8_row1", kind="mlp", fmt="int8", block=0, rows=1, d=576, ffn=1536),
        # the same of a 7B model in the smallest format: ordinary batch-1 decode
        dict(name="mlp_7b_int4_row1", kind="mlp", fmt="int4", block=32, rows=1, d=4096, ffn=11008),
        # six sequences decoded together
        dict(name="mlp_7b_int8_rows6", kind="mlp", fmt="int8", block=0, rows=6, d=4096, ffn=11008),
        # a full shared step of a ragged batch: decode rows and prompt tokens side by side
        dict(name="mlp_1b_bf16_rows13", kind="mlp", fmt="bf16", block=0, rows=13, d=2048, ffn=8192),
        # a short prompt (a chat turn) in one chunk
        dict(name="mlp_7b_bf16_rows127", kind="mlp", fmt="bf16", block=0, rows=127, d=4096, ffn=11008),
        # a chunk of a long prompt
        dict(name="mlp_7b_int4_rows1001", kind="mlp", fmt="int4", block=32, rows=1001, d=4096, ffn=11008),
        # attention of a decode step early in a conversation
        dict(name="attn_7b_bf16_ctx301", kind="attn", fmt="bf16", block=0, heads=32, kv=32, hd=128,
             ctx=301, window=0, api="fused"),
        # attention of a grouped-query model deep in a long document
        dict(name="attn_gqa_int8_ctx16001", kind="attn", fmt="int8", block=0, heads=32, kv=8, hd=128,
             ctx=16001, window=0, api="steps"),
        # the end of a sampled token with the OLMo-3 preset
        dict(name="head_7b_bf16_olmo3", kind="head", fmt="bf16", block=0, vocab=100278, d=4096,
             pick="olmo3"),
        # loading: one gate or up matrix of a bf16 checkpoint into int4 residency
        dict(name="quant_7b_int4", kind="quant", fmt="int4", block=32, src="bf16", rows=11008, cols=4096),
        # a long prompt through a whole 7B model up to its first logits
        dict(name="model_7b_int8_prompt2047", kind="model", preset="olmo3_actual_7b", fmt="int8",
             block=32, prompt=2047, steps=1),
        # short prompt, then decode token by token, on a pre-norm grouped-query 1B model
        dict(name="model_1b_bf16_decode16", kind="model", preset="llama32_1b", fmt="bf16", block=32,
             prompt=9, steps=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(v, m):
    return max(m, (v + m // 2) // m * m)


def draw(rng):
    kind = rng.choice(["mlp"] * 8 + ["attn"] * 5 + ["head"] * 2 + ["quant"] * 2 + ["model"] * 3)
    fmt = rng.choice(["bf16", "int8", "int4"])
    block = rng.choice([32, 32, 64, 128]) if fmt == "int4" else 0
    if kind == "mlp":
        rows = rng.choice([1, rng.randint(2, 8), rng.randint(9, 16), _log(rng, 17, 1024), _log(rng, 17, 1024)])
        # what the entry points take: 128-wide inner dimensions for prompt chunks, 32 for batches;
        # one row takes any (a ragged inner dimension now and then)
        m = 128 if rows > 16 or fmt == "int4" else 32
        d, ffn = _mult(_log(rng, 512, 5120), m), _mult(_log(rng, 1024, 13824), m)
        if rows == 1 and fmt != "int4" and rng.random() < 0.25:
            ffn -= rng.randint(1, 31)
        return dict(kind=kind, fmt=fmt, block=block, rows=rows, d=d, ffn=ffn)
    if kind == "attn":
        hd = rng.choice([64, 128, 128])
        kv = rng.choice([4, 8, 16, 32])
        heads = min(32, kv * rng.choice([1, 2, 4, 8]))
        ctx = _log(rng, 2, 16384 if kv <= 8 else 4096)
        window = rng.choice([0, 0, _log(rng, 64, 4096)])
        return dict(kind=kind, fmt=fmt, block=block, heads=heads, kv=kv, hd=hd, ctx=ctx, window=window,
                    api=rng.choice(["fused", "fused", "steps"]))
    if kind == "head":
        return dict(kind=kind, fmt=fmt, block=block, vocab=_log(rng, 8001, 128256),
                    d=_mult(_log(rng, 512, 4096), 128), pick=rng.choice(["greedy", "olmo3", "default"]))
    if kind == "quant":
        fmt = rng.choice(["int8", "int4"])
        return dict(kind=kind, fmt=fmt, block=rng.choice([32, 64, 128]) if fmt == "int4" else 0,
                    src=rng.choice(["bf16", "f32"]), rows=_log(rng, 257, 16384), cols=_mult(_log(rng, 512, 8192), 128))
    preset = rng.choice(["olmo3_1b", "llama32_1b", "olmo3_actual_7b"])
    return dict(kind=kind, preset=preset, fmt=fmt, block=32,
                prompt=_log(rng, 1, 700 if preset == "olmo3_actual_7b" else 1500), steps=rng.randint(1, 6))


# ---- inputs ----------------------------------------------------------------------


def _gen(seed, *salt):
    s = seed & 0x7FFFFFFF
    for v in salt:
        s = (s * 1000003 + v + 1) & 0x7FFFFFFFFFFF
    return torch.Generator(device=DEV).manual_seed(s)


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).mul_(std)


def _acts(g, rows, d):
    return _normal(g, (rows, d)) * torch.exp(_normal(g, (d,), 0.7))


def _norm_w(g, n):
    return torch.rand(n, generator=g, device=DEV).add_(0.5)


def _round_away(v):
    t = v.trunc()
    return t + ((v - t).abs() >= 0.5) * torch.sign(v)


def _quantise(w, fmt, block):
    """(stored data, scales) of an f32 matrix in a weight format (a tensor divisor: a division by a
    Python number is a product with its reciprocal, an ulp off the formats' rule)."""
    if fmt == "bf16":
        return w.to(torch.bfloat16), None
    if fmt == "int8":
        mx = w.abs().amax(1)
        s = torch.where(mx > 0, mx / torch.full_like(mx, 127.0), torch.ones_like(mx))
        return _round_away((w * (1.0 / s)[:, None]).clamp(-127, 127)).to(torch.int8), s
    b = w.reshape(-1, block)
    mx = b.abs().amax(1)
    s = torch.where(mx > 0, mx / torch.full_like(mx, 7.0), torch.ones_like(mx))
    q = _round_away((b * (1.0 / s)[:, None]).clamp(-7, 7)).to(torch.int32).reshape(-1, 2)
    return ((q[:, 0] & 15) << 4 | (q[:, 1] & 15)).to(torch.uint8), s


def _weights(g, rows, cols, fmt, block, std=0.02):
    return _quantise(_normal(g, (rows, cols), std), fmt, block)


def _dequant64(stored, rows, cols, fmt, block):
    data, s = stored
    if fmt == "bf16":
        return data.double()
    if fmt == "int8":
        return data.double() * s.double()[:, None]
    b = data.to(torch.int32)
    q = torch.stack([b >> 4, b & 15], 1).reshape(-1, block)
    q = torch.where(q >= 8, q - 16, q)
    return (q.double() * s.double()[:, None]).reshape(rows, cols)


def _ptr(t):
    return None if t is None else t.data_ptr()


def _rope(freqs, n):
    """cos and sin tables [n][len(freqs)]: the angle is an f32 product, as everywhere in this family."""
    a = (np.arange(n, dtype=np.float32)[:, None] * freqs[None, :]).astype(np.float64)
    return np.cos(a), np.sin(a)


def _freqs(theta, hd):
    i = np.arange(hd // 2, dtype=np.float32)
    e = (np.float32(2.0) * i / np.float32(hd)).astype(np.float64)
    return (np.float32(1.0) / np.power(float(theta), e).astype(np.float32)).astype(np.float32)


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


# ---- mlp ---------------------------------------------------------------------------


def _mlp_inputs(c, seed):
    g = _gen(seed, 1)
    x = _acts(g, c["rows"], c["d"])
    gu = _weights(g, 2 * c["ffn"], c["d"], c["fmt"], c["block"])
    down = _weights(g, c["d"], c["ffn"], c["fmt"], c["block"])
    return x, gu, down, _norm_w(g, c["d"])


def _mlp_prepare(c, seed):
    x, gu, down, nw = _mlp_inputs(c, seed)
    n, d, f = c["rows"], c["d"], c["ffn"]
    h = torch.empty((n, f), device=DEV)
    y, out = torch.empty((n, d), device=DEV), torch.empty((n, d), device=DEV)
    lib, fmt, blk = _lib.load(), FMT[c["fmt"]], c["block"]
    if n == 1:
        calls = [(lib.atlas_gemv_swiglu_f32, (fmt, _ptr(gu[0]), _ptr(gu[1]), blk, _ptr(x), _ptr(h), f, d)),
                 (lib.atlas_gemv_f32, (fmt, _ptr(down[0]), _ptr(down[1]), blk, _ptr(h), _ptr(y), d, f))]
    else:
        calls = [(lib.atlas_gemm_skinny_swiglu_f32,
                  (fmt, _ptr(gu[0]), _ptr(gu[1]), blk, _ptr(x), _ptr(h), f, n, d)),
                 (lib.atlas_gemm_skinny_f32,
                  (fmt, _ptr(down[0]), _ptr(down[1]), blk, _ptr(h), _ptr(y), d, n, f))]
    calls.append((lib.atlas_rmsnorm_rows_f32, (_ptr(y), _ptr(nw), _ptr(out), d, n, EPS)))
    return dict(calls=calls, keep=(x, gu, down, nw), outputs=dict(h=h, y=y, out=out))


def _mlp_exact(c, seed):
    x, gu, down, nw = _mlp_inputs(c, seed)
    d, f = c["d"], c["ffn"]
    r = x.double() @ _dequant64(gu, 2 * f, d, c["fmt"], c["block"]).t()
    gate, up = r[:, 0::2], r[:, 1::2]
    h = gate / (1.0 + torch.exp(-gate)) * up
    y = h @ _dequant64(down, d, f, c["fmt"], c["block"]).t()
    return dict(h=h, y=y, out=_rms(y, nw.double(), EPS))


# ---- attn --------------------------------------------------------------------------


def _attn_inputs(c, seed):
    g = _gen(seed, 2)
    H, KV, hd, ctx = c["heads"], c["kv"], c["hd"], c["ctx"]
    d = H * hd
    x, prev = _acts(g, 1, d), _acts(g, 1, d)
    nw, qn, kn = _norm_w(g, d), _norm_w(g, H * hd), _norm_w(g, KV * hd)
    qkv = _weights(g, (H + 2 * KV) * hd, d, c["fmt"], c["block"])
    wo = _weights(g, d, d, c["fmt"], c["block"])
    # cached keys are normalised per head and rotated: unit mean square; values as projected
    kc, vc = _normal(g, (ctx, KV, hd)), _normal(g, (ctx, KV, hd), 1.5)
    cs, sn = _rope(_freqs(500000.0, hd), ctx)
    cs, sn = (torch.from_numpy(t.astype(np.float32)).to(DEV) for t in (cs, sn))
    return x, prev, nw, qn, kn, qkv, wo, kc, vc, cs, sn


def _attn_prepare(c, seed):
    x, prev, nw, qn, kn, qkv, wo, kc, vc, cs, sn = _attn_inputs(c, seed)
    H, KV, hd, pos = c["heads"], c["kv"], c["hd"], c["ctx"] - 1
    d, m = H * hd, (H + 2 * KV) * hd
    xo, q = torch.empty((1, d), device=DEV), torch.empty((1, m), device=DEV)
    o, y = torch.empty((1, d), device=DEV), torch.empty((1, d), device=DEV)
    lib, fmt, blk = _lib.load(), FMT[c["fmt"]], c["block"]
    scale = 1.0 / math.sqrt(hd)
    calls = [(lib.atlas_gemv_fused_f32, (fmt, _ptr(qkv[0]), _ptr(qkv[1]), blk, _ptr(x), _ptr(q), m, d, 1,
                                         _ptr(prev), _ptr(nw), EPS, _ptr(xo)))]
    if c["api"] == "fused":
        calls.append((lib.atlas_attention_fused_f32,
                      (_ptr(q), _ptr(qn), _ptr(kn), EPS, _ptr(cs), _ptr(sn), _ptr(kc), _ptr(vc), _ptr(o),
                       H, KV, hd, pos, scale, c["window"], 0, 0)))
    else:
        calls += [(lib.atlas_qkv_post_f32, (_ptr(q), _ptr(qn), _ptr(kn), EPS, _ptr(cs), _ptr(sn), _ptr(kc),
                                            _ptr(vc), H, KV, hd, pos)),
                  (lib.atlas_decode_attention, (_ptr(q), _ptr(kc), _ptr(vc), _ptr(o), H, KV, hd, pos, scale,
                                                c["window"]))]
    calls.append((lib.atlas_gemv_f32, (fmt, _ptr(wo[0]), _ptr(wo[1]), blk, _ptr(o), _ptr(y), d, d)))
    return dict(calls=calls, keep=(x, prev, nw, qn, kn, qkv, wo, cs, sn, q),
                outputs=dict(x=xo, attn=o, y=y, k=kc, v=vc))


def _rotate(x, cs, sn):
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * cs - b * sn, a * sn + b * cs], -1)


def _attn_exact(c, seed):
    x, prev, nw, qn, kn, qkv, wo, kc, vc, cs, sn = _attn_inputs(c, seed)
    H, KV, hd, pos = c["heads"], c["kv"], c["hd"], c["ctx"] - 1
    d, m = H * hd, (H + 2 * KV) * hd
    xo = x.double() + _rms(prev.double(), nw.double(), EPS)
    r = xo @ _dequant64(qkv, m, d, c["fmt"], c["block"]).t()
    cs, sn = cs.double()[pos], sn.double()[pos]
    q = _rotate(_rms(r[0, :d].view(H, hd), qn.double().view(H, hd), EPS), cs, sn)
    k = _rotate(_rms(r[0, d:d + KV * hd].view(KV, hd), kn.double().view(KV, hd), EPS), cs, sn)
    kc, vc = kc.double(), vc.double()
    kc[pos], vc[pos] = k, r[0, d + KV * hd:].view(KV, hd)
    lo = max(0, pos - c["window"] + 1) if c["window"] > 0 else 0
    s = torch.einsum("kgd,tkd->kgt", q.view(KV, H // KV, hd), kc[lo:]) / math.sqrt(hd)
    o = torch.einsum("kgt,tkd->kgd", torch.softmax(s, -1), vc[lo:]).reshape(1, d)
    return dict(x=xo, attn=o, y=o @ _dequant64(wo, d, d, c["fmt"], c["block"]).t(), k=kc, v=vc)


# ---- head --------------------------------------------------------------------------


def _head_inputs(c, seed):
    g = _gen(seed, 3)
    return _acts(g, 1, c["d"]), _norm_w(g, c["d"]), _weights(g, c["vocab"], c["d"], c["fmt"], c["block"], 0.05)


def _sampling(pick, vocab):
    s = am.SamplingConfig.olmo3() if pick == "olmo3" else am.SamplingConfig()
    sup = np.array([t for t in s.suppress_initial_tokens if t < vocab] or [0], np.uint32)
    n = sum(t < vocab for t in s.suppress_initial_tokens)
    return sup, _lib.SamplingC(s.temperature, s.repetition_penalty, s.repetition_window, s.frequency_penalty,
                               s.presence_penalty, s.top_p, s.top_k, s.min_p, sup.ctypes.data, n, -1, None, 0, 0)


def _head_prepare(c, seed):
    x, nw, w = _head_inputs(c, seed)
    V, d = c["vocab"], c["d"]
    logits = torch.empty(V, device=DEV)
    lib, fmt, blk = _lib.load(), FMT[c["fmt"]], c["block"]
    calls = [(lib.atlas_gemv_fused_f32, (fmt, _ptr(w[0]), _ptr(w[1]), blk, _ptr(x), _ptr(logits), V, d, 2, None,
                                         _ptr(nw), EPS, None))]
    st = dict(calls=calls, keep=(x, nw, w), outputs=dict(logits=logits))
    if c["pick"] == "greedy":
        tok = torch.empty(1, dtype=torch.int32, device=DEV)
        calls.append((lib.atlas_argmax_u32, (_ptr(logits), V, _ptr(tok))))
        st["outputs"]["token"] = tok
    else:
        hist = np.random.default_rng(seed).integers(0, V, 200).astype(np.uint32)
        st["sample"] = (hist, *_sampling(c["pick"], V), (seed * 2654435761 + 88172645463325252) | 1)
    return st


def _head_run(st):
    _run_calls(st)
    if "sample" not in st:
        return st["outputs"]
    hist, _, s, rng0 = st["sample"]
    rng, tok = C.c_uint64(rng0), C.c_uint32(0)
    logits = st["outputs"]["logits"]
    _lib.check(_lib.load().atlas_sample_device(logits.data_ptr(), logits.numel(), hist.ctypes.data, hist.size, 5,
                                               C.byref(s), C.byref(rng), C.byref(tok)))
    return dict(logits=logits, token=int(tok.value), rng=[int(rng.value >> 32), int(rng.value & 0xFFFFFFFF)])


def _head_exact(c, seed):
    x, nw, w = _head_inputs(c, seed)
    logits = _dequant64(w, c["vocab"], c["d"], c["fmt"], c["block"]) @ _rms(x.double(), nw.double(), EPS)[0]
    out = dict(logits=logits, token=None)
    return out if c["pick"] == "greedy" else dict(out, rng=None)


# ---- quant -------------------------------------------------------------------------


def _quant_inputs(c, seed):
    w = _normal(_gen(seed, 4), (c["rows"], c["cols"]), 0.02)
    return w.to(torch.bfloat16) if c["src"] == "bf16" else w


def _quant_prepare(c, seed):
    w = _quant_inputs(c, seed)
    n, lib = w.numel(), _lib.load()
    bf = 1 if c["src"] == "bf16" else 0
    if c["fmt"] == "int8":
        data, s = torch.empty(n, dtype=torch.int8, device=DEV), torch.empty(c["rows"], device=DEV)
        call = (lib.atlas_quantize_int8_dev, (_ptr(w), bf, c["rows"], c["cols"], _ptr(data), _ptr(s)))
    else:
        data = torch.empty(n // 2, dtype=torch.uint8, device=DEV)
        s = torch.empty(n // c["block"], device=DEV)
        call = (lib.atlas_quantize_int4_dev, (_ptr(w), bf, n, c["block"], _ptr(data), _ptr(s)))
    return dict(calls=[call], keep=(w,), outputs=dict(data=data, scales=s))


def _quant_exact(c, seed):
    w = _quant_inputs(c, seed).double()
    mx = w.abs().amax(1) / 127.0 if c["fmt"] == "int8" else w.reshape(-1, c["block"]).abs().amax(1) / 7.0
    return dict(data=None, scales=mx)


# ---- model -------------------------------------------------------------------------


def _config(c):
    cfg = getattr(am.ModelConfig, c["preset"])()
    cfg.max_seq_len = 4096
    if c["preset"] == "llama32_1b":          # a Llama checkpoint has neither
        cfg.post_norm = cfg.qk_norm = False
    return cfg


def _tensors(cfg, layer):
    """(kind, rows, cols or None for a norm) of one layer, or of the rest for layer -1."""
    d, kv, f = cfg.d_model, cfg.kv_dim(), cfg.ffn_hidden
    if layer < 0:
        return [(am.T_EMBED, cfg.vocab_size, d), (am.T_LM_HEAD, cfg.vocab_size, d), (am.T_FINAL_NORM, d, None)]
    t = [(am.T_WQ, d, d), (am.T_WK, kv, d), (am.T_WV, kv, d), (am.T_WO, d, d), (am.T_W_GATE, f, d),
         (am.T_W_UP, f, d), (am.T_W_DOWN, d, f), (am.T_ATTN_NORM, d, None), (am.T_FFN_NORM, d, None)]
    return t + ([(am.T_Q_NORM, d, None), (am.T_K_NORM, kv, None)] if cfg.qk_norm else [])


def _tensor(seed, kind, layer, rows, cols):
    g = _gen(seed, 5, layer + 1, kind)
    if cols is None:
        return _norm_w(g, rows)
    w = torch.empty((rows, cols), dtype=torch.bfloat16, device=DEV)
    return w.normal_(0.0, 0.02, generator=g)


def _tokens(c, cfg, seed):
    r = np.random.default_rng(seed + 77)
    return [int(t) for t in r.integers(0, cfg.vocab_size, c["prompt"] + c["steps"])]


def _model_prepare(c, seed):
    cfg = _config(c)
    m = am.OlmoModel(cfg, weight_format=FMT[c["fmt"]], int4_block=c["block"])
    lib = _lib.load()
    scratch = lib.atlas_load_scratch_create()
    for layer in range(-1, cfg.n_layers):
        held = []
        for kind, rows, cols in _tensors(cfg, layer):
            held.append((kind, _tensor(seed, kind, layer, rows, cols)))
        torch.cuda.synchronize()             # the model's stream is its own
        for kind, t in held:
            _lib.check(lib.atlas_model_set_tensor_dev(m._h, kind, max(layer, 0), t.data_ptr(),
                                                      0 if t.dtype == torch.float32 else 1, t.numel(), scratch))
        torch.cuda.synchronize()             # before this layer's sources are freed
    lib.atlas_load_scratch_destroy(scratch)
    toks = _tokens(c, cfg, seed)
    return dict(model=m, prompt=toks[:c["prompt"]], steps=toks[c["prompt"]:])


def _model_run(st):
    m = st["model"]
    m.reset()
    m.prefill(st["prompt"])
    return dict(logits=np.stack([m.forward_one(t) for t in st["steps"]]))


def _model_exact(c, seed):
    cfg = _config(c)
    V, d, H, KV, hd = cfg.vocab_size, cfg.d_model, cfg.n_heads, cfg.n_kv_heads, cfg.head_dim()
    eps = cfg.rms_norm_eps
    toks = _tokens(c, cfg, seed)
    T = len(toks)

    def mat(kind, layer, rows, cols):
        w = _tensor(seed, kind, layer, rows, cols)
        if kind == am.T_EMBED or cols is None:
            return w.double()
        return _dequant64(_quantise(w.float(), c["fmt"], c["block"]), rows, cols, c["fmt"], c["block"])

    freqs, yarn = _freqs(cfg.rope_theta, hd), cfg.rope_scaling
    if yarn:
        two_pi = np.float32(2.0) * np.float32(math.pi)
        low = np.float32(yarn.orig_max_pos) / (two_pi * np.float32(yarn.beta_slow))
        high = np.float32(yarn.orig_max_pos) / (two_pi * np.float32(yarn.beta_fast))
        wl, fac = two_pi / freqs, np.float32(yarn.factor)
        a = ((wl - high) / (low - high)).astype(np.float32)
        mid = freqs / (a * fac + (np.float32(1.0) - a))
        freqs = np.where(wl < high, freqs, np.where(wl > low, freqs / fac, mid)).astype(np.float32)
    scale = (yarn.attn_factor if yarn else 1.0) / math.sqrt(hd)
    cs, sn = (torch.from_numpy(t).to(DEV)[:, None, :] for t in _rope(freqs, T))
    rest = {k: mat(k, -1, r, cc) for k, r, cc in _tensors(cfg, -1) if k != am.T_LM_HEAD}
    x = rest[am.T_EMBED][torch.tensor(toks, device=DEV)]
    fnorm = rest[am.T_FINAL_NORM]
    del rest
    t = torch.arange(T, device=DEV)
    for layer in range(cfg.n_layers):
        W = {k: mat(k, layer, r, cc) for k, r, cc in _tensors(cfg, layer)}
        xin = x if cfg.post_norm else _rms(x, W[am.T_ATTN_NORM], eps)
        q, k, v = ((xin @ W[n].t()).view(T, -1, hd) for n in (am.T_WQ, am.T_WK, am.T_WV))
        if cfg.qk_norm:
            q = _rms(q, W[am.T_Q_NORM].view(H, hd), 1e-6)
            k = _rms(k, W[am.T_K_NORM].view(KV, hd), 1e-6)
        q, k = _rotate(q, cs, sn), _rotate(k, cs, sn)
        seen = t[None, :] <= t[:, None]
        if cfg.sliding_window and layer < len(cfg.layer_types) and cfg.layer_types[layer] == "sliding":
            seen &= t[None, :] > t[:, None] - cfg.sliding_window
        o = torch.empty_like(q)
        for h in range(H):
            s = (q[:, h] @ k[:, h * KV // H].t()) * scale
            o[:, h] = torch.softmax(s.masked_fill_(~seen, -math.inf), -1) @ v[:, h * KV // H]
        a = o.view(T, d) @ W[am.T_WO].t()
        x = x + (_rms(a, W[am.T_ATTN_NORM], eps) if cfg.post_norm else a)
        xin = x if cfg.post_norm else _rms(x, W[am.T_FFN_NORM], eps)
        gate = xin @ W[am.T_W_GATE].t()
        f = (gate / (1.0 + torch.exp(-gate)) * (xin @ W[am.T_W_UP].t())) @ W[am.T_W_DOWN].t()
        x = x + (_rms(f, W[am.T_FFN_NORM], eps) if cfg.post_norm else f)
        del W
    x = _rms(x[-c["steps"]:], fnorm, eps)
    return dict(logits=x @ mat(am.T_LM_HEAD, -1, V, d).t())


# ---- the five kinds ----------------------------------------------------------------


def _run_calls(st):
    for fn, args in st["calls"]:
        rc = fn(*args)
        if rc is not None and rc < 0:
            _lib.check(rc)
    return st["outputs"]


_PREPARE = dict(mlp=_mlp_prepare, attn=_attn_prepare, head=_head_prepare, quant=_quant_prepare, model=_model_prepare)
_EXACT = dict(mlp=_mlp_exact, attn=_attn_exact, head=_head_exact, quant=_quant_exact, model=_model_exact)


def prepare(case, seed):
    st = _PREPARE[case["kind"]](case, seed)
    st["run"] = {"head": _head_run, "model": _model_run}.get(case["kind"], _run_calls)
    return st


def run(state):
    return state["run"](state)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _stored_bytes(rows, cols, fmt, block):
    n = rows * cols
    return 2 * n if fmt == "bf16" else n + 4 * rows if fmt == "int8" else n // 2 + 4 * (n // block)


def work(case):
    c, fmt, blk = case, case["fmt"], case["block"]
    if c["kind"] == "mlp":
        n, d, f = c["rows"], c["d"], c["ffn"]
        wb = _stored_bytes(2 * f, d, fmt, blk) + _stored_bytes(d, f, fmt, blk)
        return dict(bytes=wb + 4 * (3 * n * d + n * f + d), flops=6.0 * n * d * f)
    if c["kind"] == "attn":
        H, KV, hd, ctx = c["heads"], c["kv"], c["hd"], c["ctx"]
        d, m = H * hd, (H + 2 * KV) * hd
        span = min(ctx, c["window"]) if c["window"] > 0 else ctx
        wb = _stored_bytes(m, d, fmt, blk) + _stored_bytes(d, d, fmt, blk)
        return dict(bytes=wb + 4 * (2 * span * KV * hd + 6 * d + 2 * m), flops=2.0 * m * d + 2.0 * d * d + 4.0 * span * d)
    if c["kind"] == "head":
        return dict(bytes=_stored_bytes(c["vocab"], c["d"], fmt, blk) + 4 * (c["vocab"] + 2 * c["d"]),
                    flops=2.0 * c["vocab"] * c["d"])
    if c["kind"] == "quant":
        n = c["rows"] * c["cols"]
        return dict(bytes=n * (2 if c["src"] == "bf16" else 4) + _stored_bytes(c["rows"], c["cols"], fmt, blk),
                    flops=2.0 * n)
    cfg = _config(c)
    V, d, T = cfg.vocab_size, cfg.d_model, c["prompt"] + c["steps"]
    el = sum(r * k for kind, r, k in _tensors(cfg, 0) if k)
    wb = cfg.n_layers * sum(_stored_bytes(r, k, fmt, blk) for kind, r, k in _tensors(cfg, 0) if k)
    # the prompt needs the weights once, every later token again
    passes = (1 if c["prompt"] else 0) + c["steps"]
    kvb = 8 * cfg.kv_dim() * cfg.n_layers
    return dict(bytes=passes * wb + c["steps"] * (_stored_bytes(V, d, fmt, blk) + 4 * V) + kvb * (T + c["steps"] * T),
                flops=2.0 * T * el * cfg.n_layers + 2.0 * c["steps"] * V * d + 2.0 * T * T * d * cfg.n_layers)


def tolerance(case):
    # About four times what each way of computing shows against 64 bits over these ranges:
    #  * 32-bit sums in another order: up to 3.5e-7 (largest difference 1.5e-6);
    #  * activations in two bf16 parts for the matrix cores (more than one row): 9e-6 (1e-4);
    #  * int4 weights of one row in 16-bit products around an offset: 8e-5 (4e-4).
    # A whole model carries them through all its layers: 9e-6 (5e-5), with int4 weights 2.2e-4 (1e-3).
    int4 = case["fmt"] == "int4"
    if case["kind"] == "quant":
        return "exact"
    if case["kind"] == "model":
        return {"rel": 9e-4, "max": 4e-3} if int4 else {"rel": 4e-5, "max": 2e-4}
    if case["kind"] == "mlp" and case["rows"] > 1:
        return {"rel": 4e-5, "max": 4e-4}
    return {"rel": 3e-4, "max": 2e-3} if int4 else {"rel": 1.5e-6, "max": 6e-6}
