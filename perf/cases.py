"""Measured cases: what a user of this framework runs through its public entry
points, from single tokens of the smallest model to batched prompts.

Kinds:
  generate  LlamaModel.generate_greedy on one prompt (cache, prompt, token loop)
  decode    one request on a loaded model: new cache, prefill, then tokens fed
            one by one through forward_with_llama_cache, logits each
  serve     one batch of requests: new caches, batched prefill, batched decode
  layer     one Llama decoder layer over the backend trait, op by op as the
            generic model calls it: past > 0 is one cached decode token
            (llama.rs:371-468, 485-511), past == 0 a prompt (llama.rs:162-266)
  mlp       RMSNorm, gate / up, SwiGLU, down, residual over the backend trait
  block     one GPT-2 (causal) or Whisper-encoder (full attention) block:
            LayerNorm, Linear layers with bias, attention, GELU
  head      final norm, logits, next token (greedy or sampled)

`exact` restates each kind in float64 with torch alone.
"""
import math

import numpy as np
import torch

import esolearn_amd as E
import esolearn_amd.llama as EL

B = E.HipBackend
EPS = 1e-5
QMODE = {"int8": EL.QUANT_PER_TENSOR, "block32": EL.QUANT_BLOCK32, "bf16": EL.QUANT_BF16}
# (hidden, heads, KV heads, ffn, vocab, rope theta) of this repository's configurations
TINY = dict(h=288, nh=6, nkv=6, ffn=768, vocab=32000, theta=10000.0)
L7B = dict(h=4096, nh=32, nkv=32, ffn=11008, vocab=32000, theta=10000.0)
L8B = dict(h=4096, nh=32, nkv=8, ffn=14336, vocab=128256, theta=500000.0)


def listed():
    return [
        # the smallest model end to end: every step is launch-bound
        dict(name="generate_tiny", kind="generate", **TINY, layers=6, weights="int8", prompt=9, new=24),
        # chat on the 7B shape at full depth: a 512-token prompt, then tokens one by one
        dict(name="decode_7b", kind="decode", **L7B, layers=32, weights="int8", prompt=512, new=24),
        # four long prompts served together (GQA, the largest vocabulary)
        dict(name="serve_8b", kind="serve", **L8B, layers=2, weights="int8", seqs=4, prompt=1023, new=8),
        # one cached token through one layer, op by op: a long multi-head context ...
        dict(name="layer_decode_7b", kind="layer", **L7B, weights="int8", rows=1, past=1000),
        # ... and a short grouped-query one on block-32 weights
        dict(name="layer_decode_8b_b32", kind="layer", **L8B, weights="block32", rows=1, past=77),
        # a prompt through one layer, op by op
        dict(name="layer_prompt_8b", kind="layer", **L8B, weights="int8", rows=512, past=0),
        # a short ragged prompt in bf16 mode
        dict(name="layer_prompt_7b_bf16", kind="layer", **L7B, weights="bf16", rows=37, past=0),
        # the MLP at a batch between decode and prefill
        dict(name="mlp_8b_130", kind="mlp", **L8B, weights="int8", rows=130),
        # GPT-2 small, quantized Linear layers, an ordinary prompt
        dict(name="block_gpt2", kind="block", h=768, nh=12, ffn=3072, rows=200, causal=True, weights="int8"),
        # Whisper large's encoder block over 30 s of audio, unquantized
        dict(name="block_whisper_f32", kind="block", h=1280, nh=20, ffn=5120, rows=1500, causal=False, weights="f32"),
        # the largest LM head, sampled as a chat does
        dict(name="head_8b_sample", kind="head", h=4096, vocab=128256, rows=1, weights="int8", norm="rms",
             temperature=0.8, top_k=40, top_p=0.95),
        # GPT-2's tied f32 head, greedy
        dict(name="head_gpt2_f32", kind="head", h=768, vocab=50257, rows=1, weights="f32", norm="layer",
             temperature=0.0, top_k=0, top_p=1.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["generate", "decode", "serve", "layer", "layer", "layer", "layer", "mlp", "block", "block", "head", "head"])
    dims = dict(rng.choice([TINY, L7B, L8B]))
    if kind == "generate":
        return dict(kind=kind, **TINY, layers=rng.randint(1, 6), weights=rng.choice(["int8", "block32", "bf16"]),
                    prompt=_log(rng, 1, 64), new=rng.randint(4, 48))
    if kind == "decode":
        return dict(kind=kind, **dims, layers=rng.randint(1, 2), weights=rng.choice(["int8", "block32", "bf16"]),
                    prompt=_log(rng, 2, 1024), new=rng.randint(1, 16))
    if kind == "serve":
        return dict(kind=kind, **dims, layers=rng.randint(1, 2), weights=rng.choice(["int8", "int8", "block32"]),
                    seqs=rng.randint(2, 8), prompt=_log(rng, 8, 512), new=rng.randint(2, 12))
    if kind == "layer":
        if rng.random() < 0.5:
            return dict(kind=kind, **dims, weights=rng.choice(["int8", "int8", "block32", "bf16", "f32"]), rows=1,
                        past=_log(rng, 2, 2047))
        w = rng.choice(["int8", "int8", "block32", "bf16", "f32"])
        return dict(kind=kind, **dims, weights=w, rows=_log(rng, 2, 256 if w == "f32" else 1024), past=0)
    if kind == "mlp":
        return dict(kind=kind, **dims, weights=rng.choice(["int8", "int8", "block32", "bf16"]), rows=_log(rng, 1, 1024))
    if kind == "block":
        h, nh = rng.choice([(768, 12), (512, 8), (1280, 20), (384, 6)])
        causal = h == 768
        return dict(kind=kind, h=h, nh=nh, ffn=4 * h, rows=_log(rng, 1, 1024) if causal else rng.randint(100, 1500),
                    causal=causal, weights=rng.choice(["int8", "f32", "bf16"]))
    h, vocab, norm = rng.choice([(4096, 32000, "rms"), (4096, 128256, "rms"), (768, 50257, "layer"), (288, 32000, "rms")])
    t, k, p = rng.choice([(0.0, 0, 1.0), (1.0, 0, 1.0), (0.8, 40, 0.95), (0.9, 0, 0.9)])
    return dict(kind=kind, h=h, vocab=vocab, rows=1, weights=rng.choice(["int8", "int8", "f32"]), norm=norm,
                temperature=t, top_k=k, top_p=p)


# ------------------------------------------------------------------- inputs
class _Draw:
    """Seeded tensors on the GPU, the same for prepare and exact."""

    def __init__(self, seed):
        self.g = torch.Generator("cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(std).add_(mean)

    def rows(self, m, h):
        # a residual stream: a few channels carry much larger values
        x = self.normal(m, h)
        x[:, torch.randint(0, h, (4,), generator=self.g, device="cuda")] *= 12.0
        return x

    def ids(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.g, device="cuda").cpu().numpy().astype(np.int64)

    def weight(self, k, n, kind):
        """(stored values, scales) of a [k, n] weight; N(0, 0.02) as the models' init."""
        if kind in ("f32", "bf16"):
            w = self.normal(k, n, std=0.02)
            return (w.to(torch.bfloat16) if kind == "bf16" else w), None
        q = self.normal(k, n, std=23.0).round_().clamp_(-127, 127).to(torch.int8)
        if kind == "int8":
            return q, 0.02 / 23.0
        nb = (k + 31) // 32
        return q, (0.02 / 23.0) * (1.0 + 0.2 * torch.rand(n, nb, generator=self.g, device="cuda"))


class _Weight:
    """A projection in device storage, applied as the generic modules do."""

    def __init__(self, w, kind):
        v, s = w
        self.kind, (self.k, self.n) = kind, v.shape
        if kind == "f32":
            self.w = B.from_vec(v.cpu().numpy())
        elif kind == "bf16":
            bits = v.view(torch.int16).cpu().numpy().view(np.uint16)
            B.set_bf16_mode(True)
            self.w = B.from_vec_with_bf16(v.float().cpu().numpy(), bits)
            B.set_bf16_mode(False)
        else:
            self.w = B.i8_from_vec(v.cpu().numpy())
            self.s = float(np.float32(s)) if kind == "int8" else B.from_vec(s.cpu().numpy())

    def __call__(self, x, m):
        if self.kind == "int8":
            return B.matmul_i8_f32(x, self.w, self.s, m, self.k, self.n)
        if self.kind == "block32":
            return B.matmul_i8_f32_block32(x, self.w, self.s, m, self.k, self.n)
        return B.matmul(x, self.w, m, self.k, self.n)


def _wide(w):
    """A drawn weight in float64 (the value its storage stands for)."""
    v, s = w
    if s is None:
        return v.double()
    if isinstance(s, float):
        return v.double() * float(np.float32(s))
    return v.double() * s.double().repeat_interleave(32, dim=1)[:, :v.shape[0]].t()


def _vec(t):
    return B.from_vec(t.cpu().numpy())


def _freqs(c):
    hd = c["h"] // c["nh"]
    f = 1.0 / np.power(np.float64(c["theta"]), 2.0 * np.arange(hd // 2, dtype=np.float64) / hd)
    return f.astype(np.float32)


def _layer_inputs(c, seed):
    d = _Draw(seed)
    h, hd = c["h"], c["h"] // c["nh"]
    kvd = c["nkv"] * hd
    t = dict(x=d.rows(c["rows"], h), g1=d.normal(h, std=0.1, mean=1.0), g2=d.normal(h, std=0.1, mean=1.0))
    if c["kind"] == "layer":
        t["qkv"] = d.weight(h, h + 2 * kvd, c["weights"])
        t["o"] = d.weight(h, h, c["weights"])
    for n in ("gate", "up"):
        t[n] = d.weight(h, c["ffn"], c["weights"])
    t["down"] = d.weight(c["ffn"], h, c["weights"])
    if c.get("past"):
        t["k"], t["v"] = d.normal(c["past"], kvd), d.normal(c["past"], kvd)
    return t


def _block_inputs(c, seed):
    d = _Draw(seed)
    h, f = c["h"], c["ffn"]
    t = dict(x=d.rows(c["rows"], h))
    for n in ("g1", "g2"):
        t[n] = d.normal(h, std=0.1, mean=1.0)
    for n in ("b1", "b2"):
        t[n] = d.normal(h, std=0.1)
    for n, k, m in (("qkv", h, 3 * h), ("o", h, h), ("fc", h, f), ("proj", f, h)):
        t[n] = (*d.weight(k, m, c["weights"]), d.normal(m, std=0.1))
    return t


def _head_inputs(c, seed):
    d = _Draw(seed)
    t = dict(x=d.rows(c["rows"], c["h"]), g=d.normal(c["h"], std=0.1, mean=1.0), b=d.normal(c["h"], std=0.1))
    t["w"] = d.weight(c["h"], c["vocab"], c["weights"])
    return t


def _deep(c):
    return c["layers"] > 6 or (c["layers"] > 2 and c["h"] > 1024)


def _model_tensors(c, seed):
    """(tensor id, layer, [in, out] or [V, h] f32) of a shallow model, one at a time."""
    d = _Draw(seed)
    h, hd = c["h"], c["h"] // c["nh"]
    kvd = c["nkv"] * hd
    yield EL.T_EMBED, 0, d.normal(c["vocab"], h, std=0.02)
    for i in range(c["layers"]):
        for tid, k, n in ((EL.T_QKV, h, h + 2 * kvd), (EL.T_O, h, h), (EL.T_GATE, h, c["ffn"]),
                          (EL.T_UP, h, c["ffn"]), (EL.T_DOWN, c["ffn"], h)):
            yield tid, i, d.normal(k, n, std=0.02)
    yield EL.T_LM_HEAD, 0, d.normal(c["vocab"], h, std=0.02)


def _tokens(c, seed):
    d = _Draw(seed + 7)
    n = c.get("seqs", 1)
    return d.ids(n * (c["prompt"] + c["new"]), c["vocab"]).reshape(n, -1)


def prepare(case, seed):
    E.init(0)
    c, kind = case, case["kind"]
    if kind in ("generate", "decode", "serve"):
        cfg = E.LlamaConfig(c["vocab"], c["h"], c["ffn"], c["layers"], c["nh"], c["nkv"], max_seq_len=2048,
                            rope_theta=c["theta"], tie_word_embeddings=False)
        m = E.LlamaModel.new_random(cfg, seed=seed, quant_mode=QMODE[c["weights"]], init_on_device=True)
        if not _deep(c):
            for tid, layer, w in _model_tensors(c, seed):
                m.set_tensor(tid, layer, w.cpu().numpy())
        return dict(c=c, m=m, t=_tokens(c, seed))
    if kind in ("layer", "mlp"):
        t = _layer_inputs(c, seed)
        s = dict(c=c, x=_vec(t["x"]), g1=_vec(t["g1"]), g2=_vec(t["g2"]))
        for n in ("qkv", "o", "gate", "up", "down"):
            if n in t:
                s[n] = _Weight(t[n], c["weights"])
        if kind == "layer":
            s["freqs"] = B.from_vec(_freqs(c))
        if c.get("past"):
            s["max_seq"] = c["past"] + 256
            for n in ("k", "v"):
                full = torch.zeros(s["max_seq"], t[n].shape[1], device="cuda")
                full[:c["past"]] = t[n]
                s[n + "c"] = _vec(full)
        return s
    if kind == "block":
        t = _block_inputs(c, seed)
        s = dict(c=c)
        for n in ("x", "g1", "b1", "g2", "b2"):
            s[n] = _vec(t[n])
        for n in ("qkv", "o", "fc", "proj"):
            v, sc, bias = t[n]
            k, out = v.shape
            if c["weights"] == "int8":
                s[n] = (B.i8_from_vec(v.cpu().numpy()), float(np.float32(sc)), _vec(bias), k, out)
            else:
                s[n] = E.Linear(_Weight((v, sc), c["weights"]).w, _vec(bias), k, out)
        return s
    t = _head_inputs(c, seed)
    return dict(c=c, x=_vec(t["x"]), g=_vec(t["g"]), b=_vec(t["b"]),
                w=_vec(t["w"][0].t().contiguous()) if c["weights"] == "f32" else _Weight(t["w"], c["weights"]),
                cfg=E.SamplingConfig(c["temperature"], c["top_k"], c["top_p"], 1), seed=seed)


# --------------------------------------------------------------------- runs
def run(s):
    c = s["c"]
    bf16 = c["weights"] == "bf16" and c["kind"] not in ("generate", "decode", "serve")
    if bf16:
        B.set_bf16_mode(True)
    try:
        return _RUN[c["kind"]](s, c)
    finally:
        if bf16:
            B.set_bf16_mode(False)


def _run_generate(s, c):
    toks, lg = s["m"].generate_greedy(s["t"][0, :c["prompt"]], c["new"], want_logits=True)
    return {"tokens": toks, "logits": lg}


def _run_decode(s, c):
    m, t, p = s["m"], s["t"][0], c["prompt"]
    cache = m.new_llama_kv_cache(p + c["new"])
    out = []
    if p > 1:
        out.append(m.prefill([cache], t[None, :p - 1])[0])
    for i in range(c["new"]):
        out.append(m.forward_with_llama_cache(t[p - 1 + i], p - 1 + i, cache)[0])
    cache.free()
    return {"logits": out}


def _run_serve(s, c):
    m, t, p = s["m"], s["t"], c["prompt"]
    caches = [m.new_llama_kv_cache(p + c["new"]) for _ in range(c["seqs"])]
    first = m.prefill(caches, t[:, :p])
    toks, lg = m.decode_batch(caches, t[:, p], c["new"], want_logits=True)
    for k in caches:
        k.free()
    return {"prompt_logits": first, "tokens": toks, "logits": lg}


def _mlp(s, c, x):
    m, h, f = c["rows"], c["h"], c["ffn"]
    n = B.rmsnorm(x, s["g2"], m, h, EPS)
    a = B.swiglu(s["gate"](n, m), s["up"](n, m))
    return B.add(x, s["down"](a, m))


def _run_mlp(s, c):
    return _mlp(s, c, s["x"]).to_vec()


def _run_layer(s, c):
    m, h, nh, nkv = c["rows"], c["h"], c["nh"], c["nkv"]
    hd = h // nh
    kvd, past = nkv * hd, c["past"]
    scale = 1.0 / math.sqrt(hd)
    qkv = s["qkv"](B.rmsnorm(s["x"], s["g1"], m, h, EPS), m)
    w = h + 2 * kvd
    q = B.gather_columns(qkv, m, w, 0, h)
    k = B.gather_columns(qkv, m, w, h, kvd)
    v = B.gather_columns(qkv, m, w, h + kvd, kvd)
    k = B.rope_with_freqs_preloaded(k, m, nkv, hd, past, s["freqs"])
    if past:
        q = B.rope_with_freqs_scaled_preloaded(q, 1, nh, hd, past, s["freqs"], scale)
        B.scatter_rows(s["kc"], k, s["max_seq"], kvd, past, 1)
        B.scatter_rows(s["vc"], v, s["max_seq"], kvd, past, 1)
        K = B.gather_reshape_repeat_kv(s["kc"], s["max_seq"], past + 1, nkv, nh, hd)
        V = B.gather_reshape_repeat_kv(s["vc"], s["max_seq"], past + 1, nkv, nh, hd)
        p = B.softmax(B.matmul_strided_batched(q, K, nh, 1, hd, past + 1, trans_b=True), nh, past + 1)
        o = B.matmul_strided_batched(p, V, nh, 1, past + 1, hd)
    else:
        q = B.reshape_for_heads(B.rope_with_freqs_preloaded(q, m, nh, hd, 0, s["freqs"]), 1, m, nh, hd)
        K, V = B.reshape_for_heads(k, 1, m, nkv, hd), B.reshape_for_heads(v, 1, m, nkv, hd)
        if nkv != nh:
            K, V = B.repeat_kv(K, nkv, nh, m, hd), B.repeat_kv(V, nkv, nh, m, hd)
        sc = B.matmul_strided_batched(q, K, nh, m, hd, m, trans_b=True)
        B.apply_batched_causal_mask_and_scale(sc, nh, m, scale, -1e9)
        o = B.matmul_strided_batched(B.softmax(sc, nh * m, m), V, nh, m, m, hd)
    x = B.add(s["x"], s["o"](B.reshape_from_heads(o, 1, m, nh, hd), m))
    return _mlp(s, c, x).to_vec()


def _linear(l, x, m):
    if isinstance(l, E.Linear):
        return l.forward(x, m)
    return B.matmul_i8_f32_bias(x, l[0], l[1], l[2], m, l[3], l[4])


def _run_block(s, c):
    m, h, nh = c["rows"], c["h"], c["nh"]
    hd = h // nh
    n = B.layernorm_inference(s["x"], s["g1"], s["b1"], m, h, EPS)
    q, k, v = B.split_qkv_reshape_heads(_linear(s["qkv"], n, m), m, nh, hd)
    sc = B.matmul_strided_batched(q, k, nh, m, hd, m, trans_b=True)
    if c["causal"]:
        B.apply_batched_causal_mask_and_scale(sc, nh, m, 1.0 / math.sqrt(hd), -1e9)
        p = B.softmax(sc, nh * m, m)
    else:
        p = B.scaled_softmax(sc, 1.0 / math.sqrt(hd), nh * m, m)
    o = B.reshape_from_heads(B.matmul_strided_batched(p, v, nh, m, m, hd), 1, m, nh, hd)
    x = B.add(s["x"], _linear(s["o"], o, m))
    n = B.layernorm_inference(x, s["g2"], s["b2"], m, h, EPS)
    return B.add(x, _linear(s["proj"], B.gelu(_linear(s["fc"], n, m)), m)).to_vec()


def _run_head(s, c):
    h, n, m = c["h"], c["vocab"], c["rows"]
    x = B.rmsnorm(s["x"], s["g"], m, h, EPS) if c["norm"] == "rms" else B.layernorm_inference(s["x"], s["g"], s["b"], m, h, EPS)
    lg = B.matmul(x, s["w"], m, h, n, trans_b=True) if c["weights"] == "f32" else s["w"](x, m)
    tok = B.sample_token(lg, s["cfg"], E.Rng.with_seed(s["seed"]))
    return {"token": tok, "logits": lg.to_vec()}


_RUN = {"generate": _run_generate, "decode": _run_decode, "serve": _run_serve, "layer": _run_layer, "mlp": _run_mlp,
        "block": _run_block, "head": _run_head}


# -------------------------------------------------------------------- exact
def _rms(x, g):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * g


def _ln(x, g, b):
    return (x - x.mean(-1, keepdim=True)) * torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + EPS) * g + b


def _rope(x, pos0, freqs):
    # x [rows, heads, hd]: adjacent pairs rotate
    ang = torch.arange(pos0, pos0 + x.shape[0], device=x.device, dtype=torch.float64)[:, None, None] * freqs
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()), -1).reshape(x.shape)


def _attend(q, k, v, past, causal=True):
    # q [m, nh, hd]; k, v [past + m, nkv, hd] -> [m, nh * hd]
    m, nh, hd = q.shape
    rep = nh // k.shape[1]
    out = torch.empty(m, nh, hd, dtype=torch.float64, device=q.device)
    mask = torch.ones(m, past + m, dtype=torch.bool, device=q.device).tril(past) if causal else None
    for h in range(nh):
        s = (q[:, h] @ k[:, h // rep].t().contiguous()) / math.sqrt(hd)
        if mask is not None:
            s.masked_fill_(~mask, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // rep].contiguous()
    return out.reshape(m, nh * hd)


def _decoder_layer(x, w, c, freqs, past, kp, vp):
    """x [m, h]; w(name) a float64 weight; kp, vp earlier rows [past, nkv, hd]. Returns (x, k, v)."""
    h, nh, nkv = c["h"], c["nh"], c["nkv"]
    hd, m = h // nh, x.shape[0]
    kvd = nkv * hd
    qkv = _rms(x, w("g1")) @ w("qkv")
    q = _rope(qkv[:, :h].reshape(m, nh, hd), past, freqs)
    k = _rope(qkv[:, h:h + kvd].reshape(m, nkv, hd), past, freqs)
    v = qkv[:, h + kvd:].reshape(m, nkv, hd)
    if past:
        k, v = torch.cat((kp, k)), torch.cat((vp, v))
    x = x + _attend(q, k, v, past) @ w("o")
    return _mlp_exact(x, w), k, v


def _mlp_exact(x, w):
    n = _rms(x, w("g2"))
    g = n @ w("gate")
    return x + (g * torch.sigmoid(g) * (n @ w("up"))) @ w("down")


def _quantized(w, mode):
    """The [in, out] float64 value of a model weight after its layout step."""
    if mode == "bf16":
        return w.to(torch.bfloat16).double()
    # correctly rounded f32 divisions (tensor by tensor), ties away from zero:
    # one unit in a scale's last place would move a few quantized values
    if mode == "int8":
        s = w.abs().max() / torch.full((), 127.0, device="cuda")
        q = (w * (torch.ones_like(s) / s)).double()
    else:
        k, n = w.shape
        p = torch.nn.functional.pad(w, (0, 0, 0, -k % 32)).reshape(-1, 32, n)
        m = p.abs().amax(1, keepdim=True)
        s = m / torch.full_like(m, 127.0)
        q = (p * (torch.ones_like(s) / s)).double()
    q = (torch.sign(q) * torch.floor(q.abs() + 0.5)).clamp_(-127, 127) * s.double()
    return q if mode == "int8" else q.reshape(-1, n)[:k]


class _Model:
    def __init__(self, c, seed):
        self.c, self.layers = c, [{} for _ in range(c["layers"])]
        names = {EL.T_QKV: "qkv", EL.T_O: "o", EL.T_GATE: "gate", EL.T_UP: "up", EL.T_DOWN: "down"}
        one = torch.ones((), dtype=torch.float64, device="cuda")
        for tid, i, w in _model_tensors(c, seed):
            if tid == EL.T_EMBED:
                self.embed = w
            elif tid == EL.T_LM_HEAD:
                self.lm = _quantized(w.t().contiguous(), c["weights"])
            else:
                self.layers[i][names[tid]] = _quantized(w, c["weights"])
        for l in self.layers:
            l["g1"] = l["g2"] = one
        self.freqs = torch.from_numpy(_freqs(c)).cuda().double()

    def new(self):
        return [(None, None)] * len(self.layers)

    def feed(self, kv, ids, past, last=True):
        x = self.embed[torch.from_numpy(np.array(ids)).cuda()].double()
        for i, l in enumerate(self.layers):
            x, k, v = _decoder_layer(x, l.__getitem__, self.c, self.freqs, past, *kv[i])
            kv[i] = (k, v)
        x = x[-1:] if last else x
        return (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)) @ self.lm


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("generate", "decode", "serve"):
        if _deep(c):
            return None
        m, t, p = _Model(c, seed), _tokens(c, seed), c["prompt"]
        if kind == "decode":
            kv, out = m.new(), []
            if p > 1:
                out.append(m.feed(kv, t[0, :p - 1], 0)[0])
            for i in range(c["new"]):
                out.append(m.feed(kv, t[0, p - 1 + i:p + i], p - 1 + i)[0])
            return {"logits": out}
        first, logits = [], []
        for row in t:
            kv, lg = m.new(), []
            y = m.feed(kv, row[:p], 0)
            if kind == "generate":
                lg.append(y[0])
                for i in range(c["new"] - 1):
                    lg.append(m.feed(kv, [int(lg[-1].argmax())], p + i)[0])
            else:
                first.append(y[0])
                tok = int(row[p])
                for i in range(c["new"]):
                    lg.append(m.feed(kv, [tok], p + i)[0])
                    tok = int(lg[-1].argmax())
            logits.append(torch.stack(lg))
        if kind == "generate":
            return {"tokens": None, "logits": logits[0]}
        return {"prompt_logits": torch.stack(first), "tokens": None, "logits": torch.stack(logits, 1)}
    if kind in ("layer", "mlp"):
        t = _layer_inputs(c, seed)
        w = lambda n: t[n].double() if torch.is_tensor(t[n]) else _wide(t[n])  # noqa: E731
        x = t["x"].double()
        if kind == "mlp":
            return _mlp_exact(x, w).reshape(-1)
        kv = [t[n].double().reshape(c["past"], c["nkv"], -1) if c["past"] else None for n in ("k", "v")]
        return _decoder_layer(x, w, c, torch.from_numpy(_freqs(c)).cuda().double(), c["past"], *kv)[0].reshape(-1)
    if kind == "block":
        t = _block_inputs(c, seed)
        d = {n: v.double() for n, v in t.items() if torch.is_tensor(v)}
        lin = lambda n, x: x @ _wide(t[n][:2]) + t[n][2].double()  # noqa: E731
        m, h, nh = c["rows"], c["h"], c["nh"]
        q, k, v = lin("qkv", _ln(d["x"], d["g1"], d["b1"])).reshape(m, 3, nh, h // nh).unbind(1)
        x = d["x"] + lin("o", _attend(q, k, v, 0, c["causal"]))
        f = torch.nn.functional.gelu(lin("fc", _ln(x, d["g2"], d["b2"])), approximate="tanh")
        return (x + lin("proj", f)).reshape(-1)
    t = _head_inputs(c, seed)
    x = t["x"].double()
    x = _rms(x, t["g"].double()) if c["norm"] == "rms" else _ln(x, t["g"].double(), t["b"].double())
    return {"token": None, "logits": (x @ _wide(t["w"])).reshape(-1)}


# ----------------------------------------------------------- work, tolerance
def _wbytes(n, kind):
    return n * {"int8": 1.0, "block32": 1.125, "bf16": 2.0, "f32": 4.0}[kind]


def work(case):
    c = case
    h = c["h"]
    if c["kind"] == "head":
        n, m = h * c["vocab"], c["rows"]
        return {"bytes": _wbytes(n, c["weights"]) + 4.0 * m * (h + c["vocab"]), "flops": 2.0 * m * n}
    if c["kind"] == "block":
        p, m = h * 3 * h + h * h + 2 * h * c["ffn"], c["rows"]
        pairs = m * (m + 1) / 2 if c["causal"] else m * m
        return {"bytes": _wbytes(p, c["weights"]) + 8.0 * m * h, "flops": 2.0 * m * p + 4.0 * pairs * h}
    kvd = c["nkv"] * (h // c["nh"])
    mlp = 3 * h * c["ffn"]
    p = mlp + (h * (h + 2 * kvd) + h * h if c["kind"] != "mlp" else 0)
    if c["kind"] in ("layer", "mlp"):
        m, past = c["rows"], c.get("past", 0)
        pairs = (past + 1 if past else m * (m + 1) / 2) if c["kind"] == "layer" else 0
        return {"bytes": _wbytes(p, c["weights"]) + 8.0 * m * h + 8.0 * past * kvd,
                "flops": 2.0 * m * p + 4.0 * pairs * h}
    # whole models: the weights once for the prompt (token by token in
    # generate) and once per step, the K/V rows of every step read and written
    L, S, n, P, V = c["layers"], c.get("seqs", 1), c["new"], c["prompt"], c["vocab"]
    steps = n + (P - 1 if c["kind"] == "generate" else 0)
    prompt = 0 if c["kind"] == "generate" else (P if c["kind"] == "serve" else P - 1)
    ctx = sum(prompt + i + 1 for i in range(steps))
    lm = _wbytes(h * V, c["weights"])
    b = (L * _wbytes(p, c["weights"])) * (steps + (prompt > 0)) + lm * (steps + (prompt > 0))
    b += S * 8.0 * L * kvd * (ctx + prompt) + 4.0 * S * V * (n + (prompt > 0))
    tok = S * (prompt + steps)
    f = 2.0 * L * p * tok + 2.0 * h * V * S * (steps + (prompt > 0)) + 4.0 * S * L * h * (prompt * (prompt + 1) / 2 + ctx)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # against float64: f32 sums and 24-bit digit planes 2e-7 to 2e-6 per layer;
    # whole models add the prompt attention's bf16 triples (1.4e-5 in two
    # layers) and depth; bf16 operands 4e-3 per layer, 1e-2 in two
    whole = case["kind"] in ("generate", "decode", "serve")
    if case["weights"] == "bf16":
        return {"rel": 2e-2 if whole else 1e-2}
    return {"rel": (2e-4 if _deep(case) else 6e-5) if whole else 1e-5}
