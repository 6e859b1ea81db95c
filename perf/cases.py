"""The work a user of this framework has it do, as measurable cases through its public entry points.

Every case is one call (or, for the whole models, one step) that a speech or chat program makes
over and over: single attention calls, linear layers with f16 and int8 block weights, an encoder
layer, a decoder token step over a batch of windows, a language model's token step and one batch
of its prompt.  Sizes are the ones the framework's tests and benchmark use for Whisper tiny.en,
base.en and small.en and for Qwen2.5-0.5B and 1.5B, and sizes between them.

Kinds of case:
  attention  Context.attention_batch_dev: encoder (n_q = n_kv), prompt (causal, transposed keys)
             and token (n_q = 1, one key count per sequence) calls
  linear     Context.linear_epi_dev: f32 rows through f16 weights, plain, GELU or residual store
  linear_q8  Context.linear_q8w_epi_dev: f32 rows through resident int8 block weights
  encoder    Context.encoder_layer_dev: one encoder layer over a batch of windows, in place
  decoder    Decoder.step: one token for every window, all layers and the logits
  llm_step   LLM.step: one token for every sequence, the model's layers and the logits
  llm_prompt LLM.forward: one batch of a prompt over the cache so far, all layers and the logits
"""
import math

import torch

import zwhisper_amd as z
from zwhisper_amd import _lib, ops

DEVICE = "cuda:0"

# name: (layers, state width, heads)
WHISPER = {"tiny.en": (4, 384, 6), "base.en": (6, 512, 8), "small.en": (12, 768, 12)}
WHISPER_VOCAB, WHISPER_TEXT, WHISPER_AUDIO = 51864, 448, 1500
# name: (layers, width, query heads, key/value heads, MLP width)
QWEN = {"qwen2.5-0.5b": (24, 896, 14, 2, 4864), "qwen2.5-1.5b": (28, 1536, 12, 2, 8960)}
QWEN_VOCAB, QWEN_ROPE, QWEN_EPS = 151936, 1e6, 1e-6
EPILOGUES = {"none": _lib.EPI_NONE, "gelu": _lib.EPI_GELU, "add": _lib.EPI_ADD}


def listed():
    return [
        # The smallest call of all: the self-attention of one layer of a tiny.en decoder in the middle of
        # transcribing one window.  Latency is all there is to it.
        {"name": "attention_token_1", "kind": "attention", "batch": 1, "n_q": 1, "n_kv": 187, "heads": 6, "kv_heads": 6,
         "d": 64, "causal": False, "transposed": False, "ragged": False},
        # A chat server's token step: the attention of one Qwen2.5-1.5B layer for 64 sequences of unlike lengths,
        # each with its own count of cached keys.  Bound by reading the caches.
        {"name": "attention_token_64", "kind": "attention", "batch": 64, "n_q": 1, "n_kv": 4096, "heads": 12,
         "kv_heads": 2, "d": 128, "causal": False, "transposed": True, "ragged": True},
        # Bulk transcription: the attention of one base.en encoder layer over 16 windows of 30 s.
        {"name": "attention_encoder_16", "kind": "attention", "batch": 16, "n_q": 1500, "n_kv": 1500, "heads": 8,
         "kv_heads": 8, "d": 64, "causal": False, "transposed": False, "ragged": False},
        # A long prompt in one causal call over a transposed key cache (Qwen2.5-0.5B).
        {"name": "attention_prompt_2048", "kind": "attention", "batch": 1, "n_q": 2048, "n_kv": 2048, "heads": 14,
         "kv_heads": 2, "d": 64, "causal": True, "transposed": True, "ragged": False},
        # The widest projection of the same bulk transcription: base.en's MLP up with its GELU, 16 windows.
        {"name": "linear_mlp_up_16", "kind": "linear", "m": 24000, "k": 512, "n": 2048, "epilogue": "gelu"},
        # One encoder layer for a few windows at a time, as a program with some concurrent streams runs it.
        {"name": "encoder_layer_4", "kind": "encoder", "model": "base.en", "windows": 4, "frames": 1500},
        # One token of one window through one small.en decoder projection: the smallest linear call.
        {"name": "linear_q8_token_1", "kind": "linear_q8", "m": 1, "k": 768, "n": 3072, "epilogue": "gelu"},
        # The output logits of a 64-sequence Qwen2.5-1.5B token step: the longest weight stream.
        {"name": "linear_q8_logits_64", "kind": "linear_q8", "m": 64, "k": 1536, "n": 151936, "epilogue": "none"},
        # A thousand prompt tokens at once through Qwen2.5-1.5B's MLP gate: an odd number of rows.
        {"name": "linear_q8_prompt_1001", "kind": "linear_q8", "m": 1001, "k": 1536, "n": 8960, "epilogue": "none"},
        # Bulk transcription's other half: one token for each of 32 small.en windows, the whole decoder.
        {"name": "decoder_step_32", "kind": "decoder", "model": "small.en", "windows": 32},
        # A stage of two Qwen2.5-1.5B layers in a 64-sequence token step, with the embedding and the logits.
        {"name": "llm_step_64", "kind": "llm_step", "model": "qwen2.5-1.5b", "layers": 2, "sequences": 64, "n_ctx": 4096},
        # The last batch of a 2048-token prompt through the whole of Qwen2.5-0.5B.
        {"name": "llm_prompt_256", "kind": "llm_prompt", "model": "qwen2.5-0.5b", "n": 256, "past": 1792, "n_ctx": 2048},
    ]


def _log_int(rng, lo, hi):
    """A whole number of lo .. hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))))))


def draw(rng):
    kind = rng.choice(["token", "token", "encoder_attention", "prompt_attention", "linear", "linear_q8_few",
                       "linear_q8_rows", "encoder", "decoder", "llm_step", "llm_prompt"])
    if kind == "token":
        whisper = rng.random() < 0.5
        heads, kv_heads, d = rng.choice([(6, 6, 64), (8, 8, 64), (12, 12, 64)] if whisper else [(14, 2, 64), (12, 2, 128)])
        return {"kind": "attention", "batch": _log_int(rng, 1, 64), "n_q": 1, "n_kv": _log_int(rng, 16, 1500 if whisper else 4096),
                "heads": heads, "kv_heads": kv_heads, "d": d, "causal": False, "transposed": not whisper,
                "ragged": rng.random() < 0.5}
    if kind == "encoder_attention":
        heads = rng.choice([6, 8, 12])
        n = rng.choice([1500, rng.randint(100, 1500)])
        return {"kind": "attention", "batch": _log_int(rng, 1, 16 if heads <= 8 else 10), "n_q": n, "n_kv": n, "heads": heads,
                "kv_heads": heads, "d": 64, "causal": False, "transposed": rng.random() < 0.5, "ragged": False}
    if kind == "prompt_attention":
        heads, kv_heads, d = rng.choice([(14, 2, 64), (12, 2, 128)])
        n_q = _log_int(rng, 17, 2048)
        return {"kind": "attention", "batch": 1, "n_q": n_q, "n_kv": rng.randint(n_q, 2048), "heads": heads,
                "kv_heads": kv_heads, "d": d, "causal": True, "transposed": True, "ragged": False}
    if kind == "linear":
        width = rng.choice([384, 512, 768])
        k, n = rng.choice([(width, width), (width, 4 * width), (4 * width, width)])
        most = 24000 if width <= 512 else 10000
        return {"kind": "linear", "m": _log_int(rng, 100, most), "k": k, "n": n,
                "epilogue": "gelu" if n > k else rng.choice(["none", "add"])}
    if kind in ("linear_q8_few", "linear_q8_rows"):
        k, n = rng.choice([(384, 384), (512, 2048), (768, 768), (768, 3072), (3072, 768), (768, 51864), (896, 896),
                           (896, 128), (896, 4864), (4864, 896), (1536, 256), (1536, 1536), (1536, 8960), (8960, 1536)])
        if kind == "linear_q8_few":
            m = _log_int(rng, 1, 64)
        else:
            m = _log_int(rng, 65, 2048 if k * n < 8000000 else 1001) if n < 50000 else rng.randint(65, 128)
        return {"kind": "linear_q8", "m": m, "k": k, "n": n, "epilogue": rng.choice(["none", "gelu", "add"])}
    if kind == "encoder":
        model = rng.choice(["tiny.en", "base.en", "small.en"])
        return {"kind": "encoder", "model": model, "windows": _log_int(rng, 1, 16 if model != "small.en" else 8),
                "frames": rng.choice([1500, rng.randint(200, 1499)])}
    if kind == "decoder":
        return {"kind": "decoder", "model": rng.choice(["tiny.en", "base.en", "small.en"]), "windows": _log_int(rng, 1, 32)}
    if kind == "llm_step":
        return {"kind": "llm_step", "model": rng.choice(["qwen2.5-0.5b", "qwen2.5-1.5b"]), "layers": rng.randint(1, 2),
                "sequences": _log_int(rng, 1, 64), "n_ctx": rng.choice([512, 1024, 2048, 4096])}
    n = _log_int(rng, 2, 256)
    return {"kind": "llm_prompt", "model": "qwen2.5-0.5b", "n": n, "past": rng.randint(0, 2048 - 256), "n_ctx": 2048}


# ---- inputs: every tensor from the seed and a tag of its own


def _normal(seed, tag, *shape, scale=1.0):
    g = torch.Generator(device=DEVICE)
    g.manual_seed((int(seed) * 1000003 + tag) & 0x7FFFFFFFFFFFFFFF)
    t = torch.randn(shape, generator=g, device=DEVICE)
    return t if scale == 1.0 else t.mul_(scale)


def _ints(seed, tag, lo, hi, n):
    """n int32 values of lo .. hi (inclusive)."""
    g = torch.Generator(device=DEVICE)
    g.manual_seed((int(seed) * 1000003 + tag) & 0x7FFFFFFFFFFFFFFF)
    return torch.randint(lo, hi + 1, (n,), generator=g, device=DEVICE, dtype=torch.int32)


def _f16(seed, tag, n, k):
    return _normal(seed, tag, n, k, scale=k ** -0.5).to(torch.float16)


def _q8(seed, tag, n, k, scale=None):
    """Int8 block weights of a normal matrix: absmax / 127 for each 32 weights of a row."""
    w = _normal(seed, tag, n, k // 32, 32, scale=k ** -0.5 if scale is None else scale)
    amax = w.abs().amax(dim=2, keepdim=True)
    q = torch.round(w * (127.0 / amax)).to(torch.int8)
    return ops.Q8(q.reshape(n, k), (amax / 127.0).reshape(n, k // 32).contiguous(), n, k)


class _Cache:
    """One of a KVCache's buffers as an array (it keeps the cache alive)."""

    def __init__(self, kv, address, shape):
        self.kv = kv
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (address, False), "version": 2}


def _cache_tensors(kv):
    """(K, V) of a KVCache as tensors over its memory: [layer][sequence][keys][width], a transposed K
    [layer][sequence][head][dim][keys]."""
    rows = (kv.n_layer, kv.n_seq, kv.n_ctx, kv.kvw)
    kt = (kv.n_layer, kv.n_seq, kv.n_head_kv, kv.d, kv.n_ctx)
    k = torch.as_tensor(_Cache(kv, kv.info.k, kt if kv.layout == _lib.KV_KT else rows), device=DEVICE)
    return k, torch.as_tensor(_Cache(kv, kv.info.v, rows), device=DEVICE)


def _attention_inputs(c, seed):
    B, H, Hk, d, n_kv = c["batch"], c["heads"], c["kv_heads"], c["d"], c["n_kv"]
    q = _normal(seed, 1, B, c["n_q"], H * d)
    if c["transposed"]:
        k = _normal(seed, 2, B, Hk, d, (n_kv + 15) // 16 * 16)
    else:
        k = _normal(seed, 2, B, n_kv, Hk * d)
    v = _normal(seed, 3, B, n_kv, Hk * d)
    lens = _ints(seed, 4, max(1, n_kv // 4), n_kv, B) if c["ragged"] else None
    return q, k, v, lens


def _linear_inputs(c, seed):
    x = _normal(seed, 1, c["m"], c["k"])
    w = (_q8 if c["kind"] == "linear_q8" else _f16)(seed, 2, c["n"], c["k"])
    return x, w, _normal(seed, 3, c["n"], scale=0.1), _normal(seed, 4, c["m"], c["n"])


def _norm_weights(seed, tag, n):
    return _normal(seed, tag, n, scale=0.1) + 1.0


def _encoder_inputs(c, seed):
    _, ns, _ = WHISPER[c["model"]]
    w = {}
    for i, (name, n, k) in enumerate([("q_w", ns, ns), ("k_w", ns, ns), ("v_w", ns, ns), ("o_w", ns, ns),
                                      ("mlp0_w", 4 * ns, ns), ("mlp1_w", ns, 4 * ns)]):
        w[name] = _f16(seed, 10 + i, n, k)
    for i, (name, n) in enumerate([("attn_ln_b", ns), ("q_b", ns), ("v_b", ns), ("o_b", ns), ("mlp_ln_b", ns),
                                   ("mlp0_b", 4 * ns), ("mlp1_b", ns)]):
        w[name] = _normal(seed, 20 + i, n, scale=0.1)
    w["attn_ln_w"], w["mlp_ln_w"] = _norm_weights(seed, 30, ns), _norm_weights(seed, 31, ns)
    return _normal(seed, 1, c["windows"], c["frames"], ns), w


def _decoder_inputs(c, seed):
    n_layer, ns, _ = WHISPER[c["model"]]
    layers = []
    for li in range(n_layer):
        t = 1000 * (li + 1)
        w = {}
        for i, (name, n, k) in enumerate([("q_w", ns, ns), ("k_w", ns, ns), ("v_w", ns, ns), ("o_w", ns, ns),
                                          ("cq_w", ns, ns), ("ck_w", ns, ns), ("cv_w", ns, ns), ("co_w", ns, ns),
                                          ("mlp0_w", 4 * ns, ns), ("mlp1_w", ns, 4 * ns)]):
            w[name] = _q8(seed, t + i, n, k)
        for i, (name, n) in enumerate([("attn_ln_b", ns), ("q_b", ns), ("v_b", ns), ("o_b", ns), ("cross_ln_b", ns),
                                       ("cq_b", ns), ("cv_b", ns), ("co_b", ns), ("mlp_ln_b", ns), ("mlp0_b", 4 * ns),
                                       ("mlp1_b", ns)]):
            w[name] = _normal(seed, t + 50 + i, n, scale=0.1)
        for i, name in enumerate(["attn_ln_w", "cross_ln_w", "mlp_ln_w"]):
            w[name] = _norm_weights(seed, t + 80 + i, ns)
        layers.append(w)
    return {"te": _q8(seed, 1, WHISPER_VOCAB, ns, 0.05), "pe": _normal(seed, 2, WHISPER_TEXT, ns, scale=0.05),
            "ln_w": _norm_weights(seed, 3, ns), "ln_b": _normal(seed, 4, ns, scale=0.1), "layers": layers,
            "tokens": _ints(seed, 5, 0, WHISPER_VOCAB - 1, c["windows"]),
            "pos": _ints(seed, 6, 0, WHISPER_TEXT - 1, c["windows"])}


def _llm_inputs(c, seed):
    n_layer, ne, H, Hk, nff = QWEN[c["model"]]
    kvw = Hk * (ne // H)
    layers = []
    for li in range(c.get("layers", n_layer)):
        t = 1000 * (li + 1)
        w = {}
        for i, (name, n, k) in enumerate([("wq", ne, ne), ("wk", kvw, ne), ("wv", kvw, ne), ("wo", ne, ne),
                                          ("w_gate", nff, ne), ("w_up", nff, ne), ("w_down", ne, nff)]):
            w[name] = _q8(seed, t + i, n, k)
        for i, (name, n) in enumerate([("bq", ne), ("bk", kvw), ("bv", kvw)]):
            w[name] = _normal(seed, t + 50 + i, n, scale=0.1)
        for i, name in enumerate(["attn_norm", "ffn_norm"]):
            w[name] = _norm_weights(seed, t + 80 + i, ne)
        layers.append(w)
    if c["kind"] == "llm_step":
        m, pos = c["sequences"], _ints(seed, 6, c["n_ctx"] // 4, c["n_ctx"] - 1, c["sequences"])
    else:
        m, pos = c["n"], None
    return {"embd": _q8(seed, 1, QWEN_VOCAB, ne, 0.05), "output_norm": _norm_weights(seed, 3, ne), "layers": layers,
            "tokens": _ints(seed, 5, 0, QWEN_VOCAB - 1, m), "pos": pos}


def _fill(kv, seed, tag):
    k, v = _cache_tensors(kv)
    for t, at in ((k, 0), (v, 1)):
        g = torch.Generator(device=DEVICE)
        g.manual_seed((int(seed) * 1000003 + tag + at) & 0x7FFFFFFFFFFFFFFF)
        t.normal_(generator=g)
    return k, v


# ---- the cases' own interface


def prepare(case, seed):
    c = dict(case)
    ctx = ops.default_context()
    s = {"case": c, "ctx": ctx}
    kind = c["kind"]
    if kind == "attention":
        s["q"], s["k"], s["v"], s["lens"] = _attention_inputs(c, seed)
        H, Hk, d = c["heads"], c["kv_heads"], c["d"]
        s["shape"] = z.AttnShape(c["n_q"], c["n_kv"], H, Hk, d, H * d, Hk * d, H * d, c["causal"],
                                 s["k"].shape[3] if c["transposed"] else None)
        s["out"] = torch.empty_like(s["q"])
    elif kind in ("linear", "linear_q8"):
        s["x"], w, s["bias"], s["out"] = _linear_inputs(c, seed)
        s["w"] = w.resident(ctx) if kind == "linear_q8" else w
    elif kind == "encoder":
        s["x"], s["w"] = _encoder_inputs(c, seed)
        rows = c["windows"] * c["frames"]
        s["scratch"] = torch.empty(ops.encoder_layer_scratch(rows, WHISPER[c["model"]][1]), device=DEVICE)
    elif kind == "decoder":
        i = _decoder_inputs(c, seed)
        s["model"] = ops.Decoder(ctx, i["te"], i["pe"], i["ln_w"], i["ln_b"], i["layers"], WHISPER[c["model"]][2],
                                 WHISPER_TEXT, WHISPER_AUDIO, c["windows"])
        s["cache"] = _fill(s["model"].self_kv, seed, 101)
        _fill(s["model"].cross_kv, seed, 103)
        s["tokens"], s["pos"] = i["tokens"], i["pos"]
        s["logits"] = torch.empty(c["windows"], WHISPER_VOCAB, device=DEVICE)
    else:
        i = _llm_inputs(c, seed)
        _, _, H, Hk, nff = QWEN[c["model"]]
        rows = c["sequences"] if kind == "llm_step" else 1
        s["model"] = ops.LLM(ctx, i["embd"], None, i["output_norm"], i["layers"], H, Hk, nff, c["n_ctx"], rows, QWEN_ROPE,
                             QWEN_EPS)
        s["cache"] = _fill(s["model"].kv, seed, 101)
        s["tokens"], s["pos"] = i["tokens"], i["pos"]
        s["logits"] = torch.empty(rows, QWEN_VOCAB, device=DEVICE)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "attention":
        q, k, v, out = s["q"], s["k"], s["v"], s["out"]
        s["ctx"].attention_batch_dev(q, k, v, s["shape"], out, c["batch"], q.stride(0), k.stride(0), v.stride(0),
                                     out.stride(0), s["lens"])
        return out
    if kind == "linear":
        s["ctx"].linear_epi_dev(s["x"], c["m"], c["k"], s["w"], s["bias"], c["n"], s["out"], EPILOGUES[c["epilogue"]])
        return s["out"]
    if kind == "linear_q8":
        s["ctx"].linear_q8w_epi_dev(s["x"], c["m"], s["w"], s["bias"], s["out"], EPILOGUES[c["epilogue"]])
        return s["out"]
    if kind == "encoder":
        _, ns, H = WHISPER[c["model"]]
        s["ctx"].encoder_layer_dev(s["x"], c["windows"], c["frames"], ns, H, s["w"], s["scratch"])
        return s["x"]
    if kind == "llm_prompt":
        s["model"].forward(s["tokens"], c["past"], s["logits"])
    else:
        s["model"].step(s["tokens"], s["pos"], s["logits"])
    return {"logits": s["logits"], "k": s["cache"][0], "v": s["cache"][1]}


def _q8_bytes(n, k):
    return n * k + n * (k // 32) * 4


def work(case):
    c = case
    kind = c["kind"]
    if kind == "attention":
        B, n_q, n_kv, H, Hk, d = (c[x] for x in ("batch", "n_q", "n_kv", "heads", "kv_heads", "d"))
        # ragged: U[n_kv / 4, n_kv], its mean
        keys = n_kv * 0.625 if c["ragged"] else n_kv
        pairs = n_q * (n_kv - n_q) + n_q * (n_q + 1) // 2 if c["causal"] else n_q * keys
        return {"bytes": 4 * B * (2 * n_q * H * d + 2 * keys * Hk * d), "flops": 4 * B * H * d * pairs}
    if kind in ("linear", "linear_q8"):
        m, n, k = c["m"], c["n"], c["k"]
        wb = _q8_bytes(n, k) if kind == "linear_q8" else 2 * n * k
        return {"bytes": wb + 4 * (m * k + n + m * n * (2 if c["epilogue"] == "add" else 1)), "flops": 2 * m * n * k}
    if kind == "encoder":
        _, ns, _ = WHISPER[c["model"]]
        rows = c["windows"] * c["frames"]
        return {"bytes": 24 * ns * ns + 8 * rows * ns, "flops": 24 * rows * ns * ns + 4 * rows * c["frames"] * ns}
    if kind == "decoder":
        n_layer, ns, _ = WHISPER[c["model"]]
        m = c["windows"]
        per_layer = 6 * _q8_bytes(ns, ns) + 2 * _q8_bytes(4 * ns, ns)
        keys = WHISPER_TEXT / 2 + WHISPER_AUDIO
        return {"bytes": n_layer * (per_layer + 8 * m * keys * ns) + _q8_bytes(WHISPER_VOCAB, ns) + 4 * m * WHISPER_VOCAB,
                "flops": m * (n_layer * (28 * ns * ns + 4 * keys * ns) + 2 * ns * WHISPER_VOCAB)}
    n_layer, ne, H, Hk, nff = QWEN[c["model"]]
    n_layer = c.get("layers", n_layer)
    kvw = Hk * (ne // H)
    weights = ne * (2 * ne + 2 * kvw + 3 * nff)
    per_layer = _q8_bytes(2 * ne + 2 * kvw + 2 * nff, ne) + _q8_bytes(ne, nff)
    if kind == "llm_step":
        m, keys = c["sequences"], 0.625 * c["n_ctx"]
        cache, rows, pairs = 8 * m * keys * kvw, m, m * keys
    else:
        m, rows = c["n"], 1
        cache = 8 * (c["past"] + m) * kvw
        pairs = m * c["past"] + m * (m + 1) / 2
    return {"bytes": n_layer * (per_layer + cache) + _q8_bytes(QWEN_VOCAB, ne) + 4 * rows * QWEN_VOCAB,
            "flops": n_layer * (2 * m * weights + 4 * pairs * ne) + 2 * rows * ne * QWEN_VOCAB}


def tolerance(case):
    # Single calls: f32 sums (in the matrix units: split operands with f32 accumulation).  Measured against exact():
    # below 6e-7 (1.3e-6 for other attention shapes), about four times that is allowed.
    if case["kind"] in ("attention", "linear", "linear_q8"):
        return {"rel": 6e-6}
    # One layer in place (2.7e-7), and whole models, whose roundings travel through all later layers (2.7e-6 over 24).
    return {"rel": 6e-6 if case["kind"] == "encoder" else 2e-5}


# ---- the same in 64 bits, in plain torch


def _deq(w):
    return (w.q.double().reshape(w.n, -1, 32) * w.scales.double()[:, :, None]).reshape(w.n, w.k)


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _layer_norm(x, w, b, eps=1e-5):
    mean = x.mean(dim=-1, keepdim=True)
    var = ((x - mean) ** 2).mean(dim=-1, keepdim=True)
    return (x - mean) / torch.sqrt(var + eps) * w.double() + b.double()


def _rms_norm(x, w):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + QWEN_EPS) * w.double()


def _attend(q, k, v, H, causal=False, count=None):
    """One sequence: q [n_q][H d], k and v [n_kv][Hk d] of any float type; f64 [n_q][H d]."""
    d = q.shape[1] // H
    Hk = k.shape[1] // d
    n_q, n_kv = q.shape[0], k.shape[0] if count is None else int(count)
    qh = q.double().reshape(n_q, H, d).transpose(0, 1).contiguous()
    kh = k[:n_kv].double().reshape(n_kv, Hk, d).permute(1, 2, 0).contiguous()
    vh = v[:n_kv].double().reshape(n_kv, Hk, d).transpose(0, 1).contiguous()
    g = H // Hk
    out = torch.empty_like(qh)
    for j in range(Hk):
        sc = torch.matmul(qh[j * g:(j + 1) * g].reshape(g * n_q, d), kh[j]) / math.sqrt(d)
        if causal:
            see = torch.arange(n_kv, device=q.device)[None, :] <= (n_kv - n_q + torch.arange(n_q, device=q.device))[:, None]
            sc = sc.reshape(g, n_q, n_kv).masked_fill(~see, -math.inf).reshape(g * n_q, n_kv)
        out[j * g:(j + 1) * g] = torch.matmul(torch.softmax(sc, dim=-1), vh[j]).reshape(g, n_q, d)
    return out.transpose(0, 1).reshape(n_q, H * d)


def _rows(kt):
    """A transposed key cache [head][dim][keys] as rows [keys][head dim]."""
    return kt.permute(2, 0, 1).reshape(kt.shape[2], -1)


def _exact_decoder(c, seed):
    n_layer, ns, H = WHISPER[c["model"]]
    m, i = c["windows"], _decoder_inputs(c, seed)
    shape = (n_layer, m, WHISPER_TEXT, ns)
    k, v = _normal_like_fill(shape, seed, 101), _normal_like_fill(shape, seed, 102)
    ck = _normal_like_fill((n_layer, m, WHISPER_AUDIO, ns), seed, 103)
    cv = _normal_like_fill((n_layer, m, WHISPER_AUDIO, ns), seed, 104)
    k, v = k.double(), v.double()
    pos, tok = i["pos"].tolist(), i["tokens"].long()
    te = _deq(i["te"])
    x = te[tok] + i["pe"].double()[i["pos"].long()]
    each = torch.arange(m, device=DEVICE)
    for li, w in enumerate(i["layers"]):
        lin = lambda a, name: a @ _deq(w[name + "_w"]).T + (w[name + "_b"].double() if name + "_b" in w else 0.0)  # noqa: E731
        h = _layer_norm(x, w["attn_ln_w"], w["attn_ln_b"])
        q, k[li, each, i["pos"].long()], v[li, each, i["pos"].long()] = lin(h, "q"), lin(h, "k"), lin(h, "v")
        x = x + lin(torch.cat([_attend(q[j:j + 1], k[li, j], v[li, j], H, count=pos[j] + 1) for j in range(m)]), "o")
        q = lin(_layer_norm(x, w["cross_ln_w"], w["cross_ln_b"]), "cq")
        x = x + lin(torch.cat([_attend(q[j:j + 1], ck[li, j], cv[li, j], H) for j in range(m)]), "co")
        h = _gelu(lin(_layer_norm(x, w["mlp_ln_w"], w["mlp_ln_b"]), "mlp0"))
        x = x + lin(h, "mlp1")
    return {"logits": _layer_norm(x, i["ln_w"], i["ln_b"]) @ te.T, "k": k, "v": v}


def _normal_like_fill(shape, seed, tag):
    g = torch.Generator(device=DEVICE)
    g.manual_seed((int(seed) * 1000003 + tag) & 0x7FFFFFFFFFFFFFFF)
    return torch.empty(shape, device=DEVICE).normal_(generator=g)


def _rotate(x, pos, heads):
    """NeoX rotary positions: rows [n][heads d] at positions pos."""
    n, half = x.shape[0], x.shape[1] // heads // 2
    inv = QWEN_ROPE ** (-torch.arange(half, device=DEVICE, dtype=torch.float64) / half)
    ang = pos.double()[:, None] * inv
    cos, sin = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    a, b = x.reshape(n, heads, 2, half).unbind(2)
    return torch.stack([a * cos - b * sin, a * sin + b * cos], dim=2).reshape(n, -1)


def _exact_llm(c, seed):
    n_layer, ne, H, Hk, _ = QWEN[c["model"]]
    n_layer, d = c.get("layers", n_layer), ne // H
    i = _llm_inputs(c, seed)
    step = c["kind"] == "llm_step"
    n_seq, m = (c["sequences"] if step else 1), i["tokens"].numel()
    k = _normal_like_fill((n_layer, n_seq, Hk, d, c["n_ctx"]), seed, 101).double()
    v = _normal_like_fill((n_layer, n_seq, c["n_ctx"], Hk * d), seed, 102).double()
    pos = i["pos"].long() if step else c["past"] + torch.arange(m, device=DEVICE)
    at = pos.tolist()
    embd = _deq(i["embd"])
    x = embd[i["tokens"].long()]
    for li, w in enumerate(i["layers"]):
        lin = lambda a, name, b=None: a @ _deq(w[name]).T + (w[b].double() if b else 0.0)  # noqa: E731
        h = _rms_norm(x, w["attn_norm"])
        q, kk, vv = _rotate(lin(h, "wq", "bq"), pos, H), _rotate(lin(h, "wk", "bk"), pos, Hk), lin(h, "wv", "bv")
        for j in range(m):
            k[li, j if step else 0, :, :, at[j]] = kk[j].reshape(Hk, d)
            v[li, j if step else 0, at[j]] = vv[j]
        if step:
            a = torch.cat([_attend(q[j:j + 1], _rows(k[li, j]), v[li, j], H, count=at[j] + 1) for j in range(m)])
        else:
            a = _attend(q, _rows(k[li, 0]), v[li, 0], H, causal=True, count=c["past"] + m)
        x = x + lin(a, "wo")
        h = _rms_norm(x, w["ffn_norm"])
        g = lin(h, "w_gate")
        x = x + lin(g * torch.sigmoid(g) * lin(h, "w_up"), "w_down")
    last = x if step else x[-1:]
    return {"logits": _rms_norm(last, i["output_norm"]) @ embd.T, "k": k, "v": v}


def exact(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind == "attention":
        q, k, v, lens = _attention_inputs(c, seed)
        counts = lens.tolist() if lens is not None else [c["n_kv"]] * c["batch"]
        out = []
        for b in range(c["batch"]):
            kb = _rows(k[b])[:c["n_kv"]] if c["transposed"] else k[b]
            out.append(_attend(q[b], kb, v[b], c["heads"], c["causal"], counts[b]))
        return torch.stack(out)
    if kind in ("linear", "linear_q8"):
        x, w, bias, out = _linear_inputs(c, seed)
        y = x.double() @ (_deq(w) if kind == "linear_q8" else w.double()).T + bias.double()
        return _gelu(y) if c["epilogue"] == "gelu" else out.double() + y if c["epilogue"] == "add" else y
    if kind == "encoder":
        _, ns, H = WHISPER[c["model"]]
        x, w = _encoder_inputs(c, seed)
        x = x.double()
        lin = lambda a, name: a @ w[name + "_w"].double().T + (w[name + "_b"].double() if name + "_b" in w else 0.0)  # noqa: E731
        h = _layer_norm(x, w["attn_ln_w"], w["attn_ln_b"])
        q, k, v = lin(h, "q"), lin(h, "k"), lin(h, "v")
        x = x + lin(torch.stack([_attend(q[b], k[b], v[b], H) for b in range(c["windows"])]), "o")
        h = _gelu(lin(_layer_norm(x, w["mlp_ln_w"], w["mlp_ln_b"]), "mlp0"))
        return x + lin(h, "mlp1")
    return _exact_decoder(c, seed) if kind == "decoder" else _exact_llm(c, seed)
