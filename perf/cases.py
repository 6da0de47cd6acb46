"""Performance cases: the calls a user of this package makes, at the sizes they make them.

`listed()` names the fixed cases and `draw(rng)` gives more of the same ranges; `prepare` makes
what a program holds before the call (weights, caches, a decoder object, inputs), `run` is one
pass through the public entry point, `work` the bytes and operations the pass cannot do without,
`exact` the same result in 64-bit plain torch, and `tolerance` what two correct implementations of
these data types may differ by.

The kinds of case:
  audio        flash_attn_bhwd, the audio tower's self-attention (14 heads of 64): a two-second
               clip, the 30 s window and a batch of minute-long ones, bf16 and fp16
  layer        compile_kernels().decode_layer: one decoder layer of one token, as generate.py-style
               loops call it
  decode_attn  op_attention: one token's attention over a long cache
  lm_head      compile_kernels().lm_head_last: logits of the last hidden row
  decode       MegakernelPrefillDecoder.decode_step_with_logits: one token of a chat, at the start
               of a conversation and over a long context (the position is set before the call, as
               the chat.py binding does)
  fused        MegakernelFusedPrefillDecoder.prefill_step_with_logits: a short prompt, fp32
               activations
  prefill      MegakernelPrefillDecoder.prefill_step_with_logits: a prompt of 65..4096 tokens
  asr          MegakernelPrefillDecoder.prefill_asr: a prompt around a span of audio embeddings

Weights are N(0, 0.02), norm weights 1 + 0.1 N(0, 1) and tokens uniform, the distributions the
tests and bench.py use; cached keys have unit scale (they are normalised) and values the scale the
v projection of a normalised row gives.
"""
from __future__ import annotations

import math

import torch

from megaqwen_amd.chat_ops import compile_kernels
from megaqwen_amd.decoder import MegakernelFusedPrefillDecoder, MegakernelPrefillDecoder
from megaqwen_amd.flash_attn import flash_attn_bhwd

H, I, NQ, NKV, D, VOCAB = 1024, 3072, 16, 8, 128, 151936
EPS, THETA = 1e-6, 1e6
LAYER_PARAMS = (NQ + 2 * NKV) * D * H + NQ * D * H + 3 * I * H
LAYER_ROWS = (("q", NQ * D, H), ("k", NKV * D, H), ("v", NKV * D, H), ("o", H, NQ * D),
              ("gate", I, H), ("up", I, H), ("down", H, I))


def listed():
    return [
        # a two-second clip: the smallest call, host and launches count
        {"name": "audio_2s", "kind": "audio", "b": 1, "h": 14, "t": 99, "dtype": "bf16"},
        # the audio tower's full window of 30 s
        {"name": "audio_30s", "kind": "audio", "b": 1, "h": 14, "t": 1500, "dtype": "bf16"},
        # four minute-long clips at once
        {"name": "audio_batch", "kind": "audio", "b": 4, "h": 14, "t": 3000, "dtype": "fp16"},
        # one layer of a per-layer generation loop
        {"name": "decode_layer", "kind": "layer", "pos": 127, "max_seq": 4096},
        # attention of one token at the end of the longest context the model is configured for
        {"name": "decode_attn_32k", "kind": "decode_attn", "len": 32768},
        # the vocabulary projection of a per-layer generation loop
        {"name": "lm_head", "kind": "lm_head", "rows": 1},
        # a token of a chat, the whole model
        {"name": "decode_chat", "kind": "decode", "layers": 28, "pos": 200, "max_seq": 4096},
        # a token over a long context; 8 of the layers
        {"name": "decode_long", "kind": "decode", "layers": 8, "pos": 4095, "max_seq": 8192},
        # a short prompt, the whole model, fp32 activations
        {"name": "prompt_16_fused", "kind": "fused", "layers": 28, "n": 16},
        # an audio transcription prompt: 375 audio rows between text tokens; 4 layers
        {"name": "prompt_asr", "kind": "asr", "layers": 4, "n": 411, "start": 17, "audio": 375},
        # the prompt length the prefill is quoted at, the whole model
        {"name": "prompt_512", "kind": "prefill", "layers": 28, "n": 512},
        # a long prompt; 8 of the layers
        {"name": "prompt_4096", "kind": "prefill", "layers": 8, "n": 4096},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["audio", "audio", "layer", "decode_attn", "lm_head", "decode", "fused",
                       "asr", "prefill", "prefill", "prefill"])
    if kind == "audio":
        return {"kind": kind, "b": rng.choice([1, 1, 2, 3, 4]), "h": 14,
                "t": _log_int(rng, 40, 3000), "dtype": rng.choice(["bf16", "fp16"])}
    if kind == "layer":
        return {"kind": kind, "pos": _log_int(rng, 1, 4000), "max_seq": 4096}
    if kind == "decode_attn":
        return {"kind": kind, "len": _log_int(rng, 64, 32768)}
    if kind == "lm_head":
        return {"kind": kind, "rows": rng.randint(1, 64)}
    if kind == "decode":
        return {"kind": kind, "layers": rng.choice([4, 8, 16]), "pos": _log_int(rng, 1, 8000),
                "max_seq": 8192}
    if kind == "fused":
        return {"kind": kind, "layers": rng.choice([4, 8, 16, 28]), "n": rng.randint(1, 64)}
    if kind == "asr":
        audio = _log_int(rng, 50, 1500)
        start = rng.randint(4, 40)
        return {"kind": kind, "layers": rng.choice([2, 4]), "n": start + audio + rng.randint(4, 200),
                "start": start, "audio": audio}
    return {"kind": kind, "layers": rng.choice([2, 4]), "n": _log_int(rng, 65, 4096)}


# ------------------------------------------------------------------------------ inputs
def _dtype(case):
    return torch.float16 if case.get("dtype") == "fp16" else torch.bfloat16


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(gen, shape, std=1.0, dtype=torch.bfloat16):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _norm_weight(gen, n):
    return (1.0 + 0.1 * torch.randn(n, generator=gen, device="cuda")).to(torch.bfloat16)


def _layer(gen):
    """One layer's 11 tensors in the package's order: input norm, q, k, v, q norm, k norm, o,
    post norm, gate, up, down."""
    m = {k: _rand(gen, (r, c), 0.02) for k, r, c in LAYER_ROWS}
    return [_norm_weight(gen, H), m["q"], m["k"], m["v"], _norm_weight(gen, D),
            _norm_weight(gen, D), m["o"], _norm_weight(gen, H), m["gate"], m["up"], m["down"]]


def _rope(max_seq):
    """cos and sin tables [max_seq, D], each half repeated, in bf16 (built on the host, as a
    loader does)."""
    inv = 1.0 / THETA ** (torch.arange(0, D, 2, dtype=torch.float32) / D)
    f = torch.outer(torch.arange(max_seq, dtype=torch.float32), inv)
    return (torch.cos(f).repeat(1, 2).to(torch.bfloat16).cuda(),
            torch.sin(f).repeat(1, 2).to(torch.bfloat16).cuda())


def _model(gen, layers, max_seq, with_head=True):
    cos, sin = _rope(max_seq)
    return {"embed": _rand(gen, (VOCAB if with_head else 1, H), 0.02),
            "layers": [_layer(gen) for _ in range(layers)],
            "final": _norm_weight(gen, H), "cos": cos, "sin": sin}


def _cache(gen, layers, max_seq, used):
    """K and V caches [layers, NKV, max_seq, D] whose first `used` rows are filled."""
    k = torch.zeros(layers, NKV, max_seq, D, dtype=torch.bfloat16, device="cuda")
    v = torch.zeros_like(k)
    for l in range(layers):
        k[l, :, :used] = _rand(gen, (NKV, used, D))
        v[l, :, :used] = _rand(gen, (NKV, used, D), 0.64)
    return k, v


def _tokens(gen, n):
    return torch.randint(0, VOCAB, (n,), generator=gen, device="cuda").to(torch.int32).cpu()


def _inputs(case, seed):
    """The tensors of a case, from the seed alone (no object of the package)."""
    gen, kind = _gen(seed), case["kind"]
    if kind == "audio":
        shape = (case["b"], case["h"], case["t"], 64)
        return {x: _rand(gen, shape, 1.0, _dtype(case)) for x in ("q", "k", "v")}
    if kind == "layer":
        s = {"w": _layer(gen), "x": _rand(gen, (H,))}
        s["cos"], s["sin"] = _rope(case["max_seq"])
        k, v = _cache(gen, 1, case["max_seq"], case["pos"])
        s["k"], s["v"] = k[0], v[0]
        return s
    if kind == "decode_attn":
        s = _model(gen, 1, case["len"], with_head=False)
        s["k"], s["v"] = _cache(gen, 1, case["len"], case["len"])
        s["q"] = _rand(gen, (NQ * D,), 1.0, torch.float32)
        return s
    if kind == "lm_head":
        return {"h": _rand(gen, (case["rows"], H)), "norm": _norm_weight(gen, H),
                "lm": _rand(gen, (VOCAB, H), 0.02)}
    if kind == "decode":
        s = _model(gen, case["layers"], case["max_seq"])
        s["k"], s["v"] = _cache(gen, case["layers"], case["max_seq"], case["pos"])
        s["tokens"] = _tokens(gen, 1)
        return s
    s = _model(gen, case["layers"], case["n"] + 8)
    s["tokens"] = _tokens(gen, case["n"])
    if kind == "asr":
        s["audio"] = _rand(gen, (case["audio"], H), 0.02)
    return s


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    s["case"] = case
    if kind in ("layer", "lm_head"):
        s["ops"] = compile_kernels()
    if kind in ("decode_attn", "decode", "prefill", "asr", "fused"):
        cls = MegakernelFusedPrefillDecoder if kind == "fused" else MegakernelPrefillDecoder
        flat = [t for w in s["layers"] for t in w]
        n = 0 if kind in ("decode", "decode_attn") else case["n"]
        s["dec"] = cls(s["embed"], flat, s["final"], s["embed"], s["cos"], s["sin"],
                       len(s["layers"]), int(s["cos"].shape[0]), max_prefill_len=n)
        if "k" in s:
            s["dec"].get_k_cache().copy_(s["k"])
            s["dec"].get_v_cache().copy_(s["v"])
            s["k"], s["v"] = s["dec"].get_k_cache(), s["dec"].get_v_cache()
    torch.cuda.synchronize()
    return s


# -------------------------------------------------------------------------------- passes
def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "audio":
        return flash_attn_bhwd(s["q"], s["k"], s["v"])
    if kind == "layer":
        pos = case["pos"]
        y = s["ops"].decode_layer(s["x"], *s["w"], s["cos"], s["sin"], s["k"], s["v"], pos,
                                  pos + 1, case["max_seq"])
        return {"x": y, "k": s["k"][:, pos], "v": s["v"][:, pos]}
    if kind == "decode_attn":
        return s["dec"].op_attention(0, s["q"], case["len"])
    if kind == "lm_head":
        return s["ops"].lm_head_last(s["h"], s["norm"], s["lm"])
    if kind == "decode":
        pos = case["pos"]
        s["dec"].set_position(pos)
        _, logits = s["dec"].decode_step_with_logits(int(s["tokens"][0]))
        return {"logits": logits, "k": s["k"][:, :, pos], "v": s["v"][:, :, pos]}
    if kind == "asr":
        _, logits = s["dec"].prefill_asr(s["tokens"], s["audio"], case["start"],
                                         return_logits=True)
    else:
        _, logits = s["dec"].prefill_step_with_logits(s["tokens"])
    n = case["n"]
    return {"logits": logits, "k": s["dec"].get_k_cache()[:, :, :n],
            "v": s["dec"].get_v_cache()[:, :, :n]}


def work(case):
    kind = case["kind"]
    if kind == "audio":
        bh, t = case["b"] * case["h"], case["t"]
        return {"bytes": 4 * bh * t * 64 * 2, "flops": 4 * bh * t * t * 64}
    row = 2 * NKV * D * 2                                   # K and V bytes of one position
    if kind == "layer":
        n = case["pos"] + 1
        return {"bytes": 2 * LAYER_PARAMS + n * row + 4 * H,
                "flops": 2 * LAYER_PARAMS + 4 * NQ * D * n}
    if kind == "decode_attn":
        n = case["len"]
        return {"bytes": n * row + 2 * NQ * D * 4, "flops": 4 * NQ * D * n}
    if kind == "lm_head":
        return {"bytes": 2 * VOCAB * H + 2 * VOCAB, "flops": 2 * VOCAB * H}
    layers = case["layers"]
    head = 2 * VOCAB * H
    if kind == "decode":
        n = case["pos"] + 1
        return {"bytes": layers * (2 * LAYER_PARAMS + n * row) + head + 4 * VOCAB,
                "flops": layers * (2 * LAYER_PARAMS + 4 * NQ * D * n) + head}
    n = case["n"]
    return {"bytes": layers * (2 * LAYER_PARAMS + n * row) + head + 4 * VOCAB + n * 2 * H,
            "flops": layers * (2 * LAYER_PARAMS * n + 2 * NQ * D * n * (n + 1)) + head}


def tolerance(case):
    """Two correct implementations each round to the output type and, where 16-bit values pass
    between layers, differ by the roundings those carry: about twice the measured distance to the
    64-bit result."""
    kind = case["kind"]
    if kind == "audio":               # one rounding of the output (to 64 bits: 1.7e-3, 2.1e-4)
        return {"rel": 8e-4 if case["dtype"] == "fp16" else 4e-3}
    if kind == "decode_attn":         # fp32 sums in another order (to 64 bits: 3.2e-7)
        return {"rel": 2e-6}
    if kind in ("layer", "lm_head"):  # bf16 outputs of fp32 arithmetic (to 64 bits: 1.7e-3)
        return {"rel": 4e-3}
    if kind == "fused":               # bf16 cache rows of fp32 activations (to 64 bits: 1.7e-3)
        return {"rel": 4e-3}
    if kind == "decode":              # bf16 layer outputs: 0.7e-2 at 8 layers, 1.6e-2 at 28
        return {"rel": 1.5e-2 if case["layers"] <= 8 else 3.5e-2}
    # bf16 after every operation: 1e-2 at 4 layers, 1.2e-2 at 28
    return {"rel": 2.5e-2 if case["layers"] <= 8 else 3.5e-2}


# --------------------------------------------------------------------------- 64-bit results
def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(x, cos, sin):
    """rotate-half RoPE of x [..., n, D] with table rows [n, D]."""
    half = torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1)
    return x * cos.double() + half * sin.double()


def _layer64(x, w, cos, sin, past=None):
    """One decoder layer over rows x [n, H] at the positions of the table rows; `past` = (K, V) of
    the positions before, [NKV, p, D].  Returns (x', K rows, V rows)."""
    n = x.shape[0]
    ln, wq, wk, wv, qn, kn, wo, post, wg, wu, wd = w
    y = _rms(x, ln)
    q = (y @ wq.double().T).view(n, NQ, D).transpose(0, 1)
    k = (y @ wk.double().T).view(n, NKV, D).transpose(0, 1)
    v = (y @ wv.double().T).view(n, NKV, D).transpose(0, 1)
    q, k = _rotate(_rms(q, qn), cos, sin), _rotate(_rms(k, kn), cos, sin)
    kk = k if past is None else torch.cat([past[0].double(), k], 1)
    vv = v if past is None else torch.cat([past[1].double(), v], 1)
    out = torch.empty(n, NQ, D, dtype=torch.float64, device=x.device)
    keys = kk.shape[1]
    ahead = torch.arange(keys, device=x.device)[None, :] > torch.arange(
        keys - n, keys, device=x.device)[:, None]
    for h in range(NQ):
        s = (q[h] @ kk[h // (NQ // NKV)].T / math.sqrt(D)).masked_fill_(ahead, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ vv[h // (NQ // NKV)]
    x = x + out.reshape(n, NQ * D) @ wo.double().T
    y = _rms(x, post)
    g = y @ wg.double().T
    return x + (g * torch.sigmoid(g) * (y @ wu.double().T)) @ wd.double().T, k, v


def _head64(x, norm, lm):
    y = _rms(x, norm)
    return torch.cat([c.double() @ y for c in lm.split(1 << 14)])


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "audio":
        q, k, v = (s[x].double().flatten(0, 1) for x in ("q", "k", "v"))
        o = torch.stack([torch.softmax(a @ b.T / 8.0, -1) @ c for a, b, c in zip(q, k, v)])
        return o.view(s["q"].shape)
    if kind == "layer":
        p = case["pos"]
        y, k, v = _layer64(s["x"].double().view(1, H), s["w"], s["cos"][p:p + 1],
                           s["sin"][p:p + 1], (s["k"][:, :p], s["v"][:, :p]))
        return {"x": y.view(H), "k": k[:, 0], "v": v[:, 0]}
    if kind == "decode_attn":
        q, o = s["q"].double().view(NKV, NQ // NKV, D), []
        for h in range(NKV):
            a = torch.softmax(q[h] @ s["k"][0, h].double().T / math.sqrt(D), -1)
            o.append(a @ s["v"][0, h].double())
        return torch.stack(o).reshape(NQ * D)
    if kind == "lm_head":
        return _head64(s["h"][-1].double(), s["norm"], s["lm"])
    x = s["embed"][s["tokens"].cuda().long()].double()
    if kind == "asr":
        x[case["start"]:case["start"] + case["audio"]] = s["audio"].double()
    p, n, ks, vs = case.get("pos", 0), x.shape[0], [], []
    for l, w in enumerate(s["layers"]):
        past = (s["k"][l, :, :p], s["v"][l, :, :p]) if kind == "decode" else None
        x, k, v = _layer64(x, w, s["cos"][p:p + n], s["sin"][p:p + n], past)
        ks.append(k)
        vs.append(v)
    k, v = torch.stack(ks), torch.stack(vs)
    if kind == "decode":
        k, v = k[:, :, 0], v[:, :, 0]
    return {"logits": _head64(x[-1], s["final"], s["embed"]), "k": k, "v": v}
