"""Performance cases of the MiniMind decode runtime.

Each case is one call, or the short run of calls, that a program on this
runtime makes: a decoder layer for one new token or for a prompt, attention
over a cache, a projection, the vocabulary head, and whole models (a chat, a
long prompt, a batch of sequences).  Shapes are MiniMind2 and MiniMind2-small
and the 128-dimension heads of the long-context tests; `draw` spreads the same
kinds of case over their whole ranges.
"""
from __future__ import annotations

import math
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path("minimind-orangepi_amd").resolve()))

import mmr  # noqa: E402

DEVICE = "cuda"
VOCAB = 6400
THETA = 1e6
EPS = 1e-5
POSITIONS = 32768

#: hidden, layers, query heads, KV heads, head dimension, FFN width
SHAPES = {
    "minimind2": (768, 16, 8, 2, 96, 2048),
    "minimind2-small": (512, 8, 8, 2, 64, 1408),
}
HEADS = (8, 2)  # query and KV heads of every shape here


def listed():
    return [
        # A decoder layer for one token: what a program that schedules layers
        # itself calls per layer and token.  Smallest call: the small model in
        # a short chat, where launches and latency are everything.
        dict(name="layer_step_small", kind="layer_step", model="minimind2-small", position=130, kv="f16"),
        # The same in the middle of a chat, on the default fp32 cache.
        dict(name="layer_step_f32", kind="layer_step", model="minimind2", position=777, kv="f32"),
        # The same at the end of a long context, where the cache is read.
        dict(name="layer_step_long", kind="layer_step", model="minimind2", position=8190, kv="f16"),
        # Attention of one query over a resident cache, 128-dimension heads.
        dict(name="attention_d128", kind="attention", head_dim=128, tokens=4097, kv="f16"),
        # Final norm, vocabulary projection and argmax: once per token.
        dict(name="head", kind="head", hidden=768, rows=VOCAB),
        # A projection of many rows: a caller's own prompt or batch pipeline.
        dict(name="projection_rows", kind="projection", rows=4096, cols=768, batch=2048, residual=False),
        # A decoder layer over a short ragged prompt of the small model.
        dict(name="layer_prompt_small", kind="layer_prompt", model="minimind2-small", tokens=77, kv="f32"),
        # A decoder layer over an ordinary prompt.
        dict(name="layer_prompt_512", kind="layer_prompt", model="minimind2", tokens=512, kv="f16"),
        # q/k norm, RoPE, cache write and causal attention of a long prompt's
        # later part, after the rows that an earlier call has cached.
        dict(name="prompt_attention", kind="prompt_attention", head_dim=96, start=1111, tokens=3000, kv="f16"),
        # A chat turn on the whole model: prompt, then greedy decode.
        dict(name="chat", kind="model", model="minimind2", prompt=512, steps=128, kv="f16"),
        # A long document on the default fp32 cache, and the first tokens of its answer.
        dict(name="document", kind="model", model="minimind2", prompt=6000, steps=8, kv="f32"),
        # A batch of sequences, from the prompts to the last token.
        dict(name="batch", kind="batch", model="minimind2", batch=32, prompt=256, steps=16, kv="f16"),
    ]


def _between(rng, low, high):
    """A whole number in [low, high], even over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["layer_step", "layer_step", "attention", "head", "projection", "projection", "layer_prompt",
                       "layer_prompt", "prompt_attention", "chat", "document", "batch"])
    model = rng.choice(sorted(SHAPES))
    kv = rng.choice(["f16", "f32"])
    if kind == "layer_step":
        return dict(kind=kind, model=model, position=_between(rng, 16, 8191), kv=kv)
    if kind == "attention":
        return dict(kind=kind, head_dim=rng.choice([64, 96, 128]), tokens=_between(rng, 64, 8193), kv=kv)
    if kind == "head":
        return dict(kind=kind, hidden=SHAPES[model][0], rows=_between(rng, 2000, 16000))
    if kind == "projection":
        hidden, _, hq, hkv, d, ffn = SHAPES[model]
        rows, cols = rng.choice([((hq + 2 * hkv) * d, hidden), (hidden, hq * d), (2 * ffn, hidden), (hidden, ffn)])
        return dict(kind=kind, rows=rows, cols=cols, batch=_between(rng, 2, 4096), residual=rng.random() < 0.5)
    if kind == "layer_prompt":
        return dict(kind=kind, model=model, tokens=_between(rng, 5, 512), kv=kv)
    if kind == "prompt_attention":
        return dict(kind=kind, head_dim=rng.choice([64, 96, 128]), start=rng.choice([0, rng.randrange(2048)]),
                    tokens=_between(rng, 16, 4096), kv=kv)
    if kind == "chat":
        return dict(kind="model", model=model, prompt=_between(rng, 16, 1024), steps=_between(rng, 8, 128), kv=kv)
    if kind == "document":
        return dict(kind="model", model=model, prompt=_between(rng, 1024, 6000), steps=rng.randrange(1, 9), kv=kv)
    batch = _between(rng, 2, 64)
    prompt = _between(rng, 24, min(256, 8192 // batch))
    return dict(kind="batch", model=model, batch=batch, prompt=prompt, steps=rng.randrange(4, 17), kv=kv)


# ---------------------------------------------------------------- inputs ----


class Buffer:
    """Device memory of a torch tensor in the shape that mmr's calls take."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()
        self.nbytes = tensor.numel() * tensor.element_size()


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32) * std


def _weight(g, rows, cols, std=0.02):
    """A projection of a checkpoint: fp16 [rows][cols]."""
    return _normal(g, (rows, cols), std).half()


def _gain(g, n):
    return 1.0 + _normal(g, (n,), 0.1)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _kv(case):
    return (mmr.KV_F16, torch.float16) if case["kv"] == "f16" else (mmr.KV_F32, torch.float32)


def _zeros(*shape, dtype=torch.float32):
    return Buffer(torch.zeros(shape, device=DEVICE, dtype=dtype))


def _layer(g, model):
    """One layer's weights under the names of mmr.LayerWeights."""
    hidden, _, hq, hkv, d, ffn = SHAPES[model]
    return {
        "input_norm": _gain(g, hidden), "post_attention_norm": _gain(g, hidden),
        "q_norm": _gain(g, d), "k_norm": _gain(g, d),
        "q_proj": _weight(g, hq * d, hidden), "k_proj": _weight(g, hkv * d, hidden),
        "v_proj": _weight(g, hkv * d, hidden), "o_proj": _weight(g, hidden, hq * d),
        "gate_proj": _weight(g, ffn, hidden), "up_proj": _weight(g, ffn, hidden),
        "down_proj": _weight(g, hidden, ffn),
    }


def _config(model):
    hidden, layers, hq, hkv, d, ffn = SHAPES[model]
    return mmr.make_config(hidden_size=hidden, num_hidden_layers=layers, vocab_size=VOCAB, num_attention_heads=hq,
                           num_key_value_heads=hkv, head_dim=d, intermediate_size=ffn, rms_norm_eps=EPS,
                           rope_theta=THETA, max_position_embeddings=POSITIONS, tie_word_embeddings=1)


def _cache_rows(g, tokens, d, dtype):
    """Keys (normalised and rotated: about unit size) and values of a cache, [kv_head][token][d]."""
    keys, values = _normal(g, (HEADS[1], tokens, d)), _normal(g, (HEADS[1], tokens, d), 0.6)
    return keys.to(dtype), values.to(dtype)


def _cache(g, tokens, capacity, d, case):
    kv, dtype = _kv(case)
    keys, values = _cache_rows(g, tokens, d, dtype)
    cache = mmr.KvCache(HEADS[1], d, capacity, kv)
    if tokens:
        cache.upload(keys.cpu().numpy(), values.cpu().numpy())
    return cache


class _DevicePages:
    """Memory of a cache segment for torch (the CUDA array interface); a tensor of it keeps the cache."""

    def __init__(self, cache, pointer, shape, dtype):
        self.cache = cache
        self.__cuda_array_interface__ = {"data": (pointer, False), "shape": shape, "strides": None, "version": 2,
                                         "typestr": "<f2" if dtype is torch.float16 else "<f4"}


def _cache_views(cache, tokens, d, case):
    """The cache's own pages that hold positions 0 .. tokens - 1, as tensors [page][kv_head][64][d]."""
    views, s = [], 0
    while True:
        keys, values, first, held = cache.segment(s)
        if not keys or first >= tokens:
            return views
        pages = -(-(min(tokens, first + held) - first) // 64)
        for pointer in (keys, values):
            shape = (pages, HEADS[1], 64, d)
            views.append(torch.as_tensor(_DevicePages(cache, pointer, shape, _kv(case)[1]), device=DEVICE))
        s += 1


def _page_views(keys, values, tokens):
    """Full [kv_head][token][d] rows in the layout of _cache_views, zeros past the rows."""
    views, first, size = [], 0, 512
    while first < tokens:
        end = min(tokens, first + size)
        pages = -(-(end - first) // 64)
        for rows in (keys, values):
            page = rows.new_zeros((HEADS[1], pages * 64, rows.shape[-1]))
            page[:, : end - first] = rows[:, first:end]
            views.append(page.reshape(HEADS[1], pages, 64, -1).transpose(0, 1).contiguous())
        first, size = first + size, (512 if first == 0 else 2 * size)
    return views


def _model_weights(case, seed):
    """A whole model's tensors in the order of the runtime's weight file.

    A trained model is sure of most of its next tokens, which an untrained one
    is not: the tied embedding is as large as what the layers add up to, so
    greedy decoding doesn't hang on the last bits of the logits."""
    g = _generator(seed)
    hidden, layers, _, _, _, _ = SHAPES[case["model"]]
    embed = _weight(g, VOCAB, hidden, 0.5)
    tensors = [("model.embed_tokens.weight", embed), ("model.norm.weight", _gain(g, hidden)),
               ("lm_head.weight", embed)]
    for i in range(layers):
        layer = _layer(g, case["model"])
        p = "model.layers.%d." % i
        tensors += [(p + "input_layernorm.weight", layer["input_norm"]),
                    (p + "post_attention_layernorm.weight", layer["post_attention_norm"]),
                    (p + "self_attn.q_norm.weight", layer["q_norm"]), (p + "self_attn.k_norm.weight", layer["k_norm"])]
        tensors += [(p + "self_attn.%s_proj.weight" % n, layer[n + "_proj"]) for n in "qkvo"]
        tensors += [(p + "mlp.%s_proj.weight" % n, layer[n + "_proj"]) for n in ("gate", "up", "down")]
    # The file keeps every tensor in fp16, the gains too.
    return [(n, t.half()) for n, t in tensors]


def _load_model(case, seed):
    """A model from a runtime directory, as a program starts."""
    hidden, layers, hq, hkv, d, ffn = SHAPES[case["model"]]
    with tempfile.TemporaryDirectory() as folder:
        (Path(folder) / "minimind_runtime_config.txt").write_text(
            "hidden_size=%d\nnum_hidden_layers=%d\nuse_moe=0\nvocab_size=%d\nnum_attention_heads=%d\n"
            "num_key_value_heads=%d\nhead_dim=%d\nintermediate_size=%d\nmax_position_embeddings=%d\n"
            "tie_word_embeddings=1\nrms_norm_eps=%.9g\nrope_theta=%.9g\n"
            % (hidden, layers, VOCAB, hq, hkv, d, ffn, POSITIONS, EPS, THETA))
        with open(Path(folder) / "weights.bin", "wb") as f:
            f.write(b"MMRTH001")
            for name, tensor in _model_weights(case, seed):
                f.write(np.uint64(len(name)).tobytes() + name.encode() + np.uint64(tensor.numel()).tobytes())
                f.write(tensor.cpu().numpy().tobytes())
        return mmr.Model.load(folder)


def _prompts(case, seed):
    rng = np.random.default_rng(int(seed))
    if case["kind"] == "model":
        return [rng.integers(0, VOCAB, case["prompt"]).astype(np.int32)]
    # Ragged prompts: the longest as long as the case says, the shortest three quarters of it.
    lengths = [case["prompt"]] + [int(rng.integers(3 * case["prompt"] // 4, case["prompt"] + 1))
                                  for _ in range(case["batch"] - 1)]
    return [rng.integers(0, VOCAB, n).astype(np.int32) for n in lengths]


# --------------------------------------------------------------- prepare ----


def prepare(case, seed):
    return {"case": case, **_PREPARE[case["kind"]](case, seed)}


def _prepare_layer_step(case, seed):
    g = _generator(seed)
    hidden, _, _, _, d, _ = SHAPES[case["model"]]
    host = {n: t.float().cpu().numpy() for n, t in _layer(g, case["model"]).items()}
    weights = mmr.LayerWeights.create(_config(case["model"]), **host)
    cache = _cache(g, case["position"], case["position"] + 1, d, case)
    return dict(weights=weights, cache=cache, hidden=Buffer(_normal(g, (hidden,))),
                position=Buffer(torch.tensor([case["position"]], device=DEVICE, dtype=torch.int32)),
                out=_zeros(hidden), error=_zeros(1, dtype=torch.int32),
                workspace=_zeros(weights.workspace_size(512), dtype=torch.uint8),  # enough for every automatic split
                pages=_cache_views(cache, case["position"] + 1, d, case))


def _prepare_attention(case, seed):
    g = _generator(seed)
    d, tokens = case["head_dim"], case["tokens"]
    return dict(cache=_cache(g, tokens, tokens, d, case), query=Buffer(_normal(g, (HEADS[0] * d,))),
                out=_zeros(HEADS[0] * d),
                workspace=_zeros(mmr.attention_workspace_size(*HEADS, d), dtype=torch.uint8))


def _prepare_head(case, seed):
    g = _generator(seed)
    rows, hidden = case["rows"], case["hidden"]
    return dict(w=Buffer(_weight(g, rows, hidden)), x=Buffer(_normal(g, (hidden,), 3.0)), norm=Buffer(_gain(g, hidden)),
                logits=_zeros(rows), token=_zeros(1, dtype=torch.int32),
                workspace=_zeros(mmr.matvec_argmax_workspace_size(rows, hidden), dtype=torch.uint8))


def _prepare_projection(case, seed):
    g = _generator(seed)
    rows, cols, batch = case["rows"], case["cols"], case["batch"]
    return dict(w=Buffer(_weight(g, rows, cols)), x=Buffer(_normal(g, (batch, cols))), y=_zeros(batch, rows),
                residual=Buffer(_normal(g, (batch, rows))) if case["residual"] else None)


def _prepare_layer_prompt(case, seed):
    g = _generator(seed)
    hidden, _, _, _, d, _ = SHAPES[case["model"]]
    host = {n: t.float().cpu().numpy() for n, t in _layer(g, case["model"]).items()}
    weights = mmr.LayerWeights.create(_config(case["model"]), **host)
    cache = _cache(g, 0, 512, d, case)
    return dict(weights=weights, cache=cache, hidden=Buffer(_normal(g, (case["tokens"], hidden))),
                out=_zeros(case["tokens"], hidden),
                workspace=_zeros(weights.prefill_workspace_size(case["tokens"]), dtype=torch.uint8),
                pages=_cache_views(cache, case["tokens"], d, case))


def _prepare_prompt_attention(case, seed):
    g = _generator(seed)
    d, start, tokens = case["head_dim"], case["start"], case["tokens"]
    cache = _cache(g, start, start + tokens, d, case)
    return dict(cache=cache, qkv=Buffer(_normal(g, (tokens, (HEADS[0] + 2 * HEADS[1]) * d), 0.6)),
                q_norm=Buffer(_gain(g, d)), k_norm=Buffer(_gain(g, d)), rope=mmr.RopeTable(POSITIONS, d, THETA),
                query=_zeros(tokens, HEADS[0] * d), out=_zeros(tokens, HEADS[0] * d),
                pages=_cache_views(cache, start + tokens, d, case))


def _prepare_model(case, seed):
    model = _load_model(case, seed)
    state = model.make_state(case["prompt"] + case["steps"], _kv(case)[0])
    return dict(model=model, state=state, prompt=_prompts(case, seed)[0])


def _prepare_batch(case, seed):
    return dict(model=_load_model(case, seed), prompts=_prompts(case, seed))


_PREPARE = {"layer_step": _prepare_layer_step, "attention": _prepare_attention, "head": _prepare_head,
            "projection": _prepare_projection, "layer_prompt": _prepare_layer_prompt,
            "prompt_attention": _prepare_prompt_attention, "model": _prepare_model, "batch": _prepare_batch}


# ------------------------------------------------------------------- run ----


def run(state):
    return _RUN[state["case"]["kind"]](state)


def _run_layer_step(s):
    s["weights"].forward(s["cache"], s["hidden"], s["position"], s["out"], s["workspace"], 0, s["error"],
                         stream=_stream())
    return {"out": s["out"].tensor, "cache": s["pages"], "error": s["error"].tensor}


def _run_attention(s):
    c = s["case"]
    mmr.attention_from_cache(s["query"], s["cache"], c["tokens"], *HEADS, c["head_dim"], s["out"], s["workspace"],
                             stream=_stream())
    return {"out": s["out"].tensor}


def _run_head(s):
    c = s["case"]
    mmr.matvec_argmax_f16(s["w"], c["rows"], c["hidden"], s["x"], s["token"], s["workspace"], logits=s["logits"],
                          norm_w=s["norm"], eps=EPS, stream=_stream())
    return {"logits": s["logits"].tensor, "token": s["token"].tensor}


def _run_projection(s):
    c = s["case"]
    mmr.matmul_f16(s["w"], c["rows"], c["cols"], s["x"], c["batch"], s["y"], residual=s["residual"], stream=_stream())
    return {"y": s["y"].tensor}


def _run_layer_prompt(s):
    s["cache"].reset()  # a new prompt
    s["weights"].prefill(s["cache"], s["hidden"], 0, s["case"]["tokens"], s["out"], s["workspace"], stream=_stream())
    return {"out": s["out"].tensor, "cache": s["pages"]}


def _run_prompt_attention(s):
    c = s["case"]
    mmr.prefill_qkv_rows(s["qkv"], s["q_norm"], s["k_norm"], EPS, s["rope"], s["cache"], c["start"], c["tokens"],
                         *HEADS, c["head_dim"], s["query"], stream=_stream())
    mmr.prefill_attention(s["query"], s["cache"], c["start"], c["tokens"], *HEADS, c["head_dim"], s["out"],
                          stream=_stream())
    return {"query": s["query"].tensor, "out": s["out"].tensor, "cache": s["pages"]}


def _run_model(s):
    c, state = s["case"], s["state"]
    state.reset()  # a new conversation
    state.enqueue_prefill(s["prompt"])
    state.enqueue_decode(c["steps"])
    return {"logits": state.read_logits(), "tokens": state.read_sequence(c["prompt"], c["steps"] + 1)}


def _run_batch(s):
    c, prompts = s["case"], s["prompts"]
    state = s["model"].make_batch_state(len(prompts), c["prompt"] + c["steps"], _kv(c)[0])
    state.prefill(prompts)
    state.decode(c["steps"])
    logits = np.stack([state.read_logits(i) for i in range(len(prompts))])
    total = c["prompt"] + c["steps"] + 1
    tokens = np.stack([state.read_sequence(i, 0, total) for i in range(len(prompts))])
    state.free()
    return {"logits": logits, "tokens": tokens}


_RUN = {"layer_step": _run_layer_step, "attention": _run_attention, "head": _run_head, "projection": _run_projection,
        "layer_prompt": _run_layer_prompt, "prompt_attention": _run_prompt_attention, "model": _run_model,
        "batch": _run_batch}


# ------------------------------------------------------------------ work ----


def _layer_parameters(model):
    hidden, _, hq, hkv, d, ffn = SHAPES[model]
    return (hq + 2 * hkv) * d * hidden + hidden * hq * d + 3 * ffn * hidden


def _attention_flops(start, tokens, d):
    """q k and p v of `tokens` causal queries from position `start` on."""
    pairs = tokens * start + tokens * (tokens + 1) / 2
    return 4 * pairs * HEADS[0] * d


def work(case):
    kind = case["kind"]
    element = 2 if case.get("kv") == "f16" else 4
    if kind == "layer_step":
        hidden, _, _, hkv, d, _ = SHAPES[case["model"]]
        p, keys = _layer_parameters(case["model"]), case["position"] + 1
        return {"bytes": 2 * p + 2 * keys * hkv * d * element + 8 * hidden + 4 * (2 * hidden + 2 * d),
                "flops": 2 * p + _attention_flops(case["position"], 1, d)}
    if kind == "attention":
        d, tokens = case["head_dim"], case["tokens"]
        return {"bytes": 2 * tokens * HEADS[1] * d * element + 8 * HEADS[0] * d,
                "flops": _attention_flops(tokens - 1, 1, d)}
    if kind == "head":
        return {"bytes": 2 * case["rows"] * case["hidden"] + 8 * case["hidden"] + 4 * case["rows"] + 4,
                "flops": 2 * case["rows"] * case["hidden"]}
    if kind == "projection":
        rows, cols, batch = case["rows"], case["cols"], case["batch"]
        return {"bytes": 2 * rows * cols + 4 * batch * (cols + rows * (2 if case["residual"] else 1)),
                "flops": 2 * batch * rows * cols}
    if kind == "layer_prompt":
        hidden, _, _, hkv, d, _ = SHAPES[case["model"]]
        p, tokens = _layer_parameters(case["model"]), case["tokens"]
        return {"bytes": 2 * p + 2 * tokens * hkv * d * element + 8 * tokens * hidden,
                "flops": 2 * tokens * p + _attention_flops(0, tokens, d)}
    if kind == "prompt_attention":
        d, start, tokens = case["head_dim"], case["start"], case["tokens"]
        # qkv in; query and out written; the cache read up to `start`, and its new rows written.
        return {"bytes": 4 * tokens * (3 * HEADS[0] + 2 * HEADS[1]) * d + 2 * (start + tokens) * HEADS[1] * d * element,
                "flops": _attention_flops(start, tokens, d)}
    hidden, layers, _, hkv, d, _ = SHAPES[case["model"]]
    p = layers * _layer_parameters(case["model"])
    sequences = case.get("batch", 1)
    prompt, steps = case["prompt"], case["steps"]
    row = 2 * layers * hkv * d * element  # a position's keys and values
    read = sum(prompt + i + 1 for i in range(steps)) * row
    # Weights once for the prompts and once for each step; the vocabulary head once for each prediction.
    return {"bytes": (steps + 1) * 2 * (p + VOCAB * hidden) + sequences * (prompt * row + read),
            "flops": sequences * (2 * (prompt + steps) * p + 2 * (steps + 1) * VOCAB * hidden
                                  + layers * _attention_flops(0, prompt + steps, d))}


def tolerance(case):
    """About four times the distance from `exact` that was measured over the listed and drawn cases.

    On an fp32 cache everything is sums in 32 bits (single calls 0.5 to 4.5e-7, whole models to 1e-6).  On an fp16
    cache a sum that lands on the other side of a rounding boundary moves a stored key or value by 2^-10 of itself:
    rel 1e-5 over a cache, 7e-6 in attention over it, 2 to 5e-5 in a model's logits."""
    whole = case["kind"] in ("model", "batch")
    if case.get("kv") == "f16":
        return {"rel": 2e-4, "max": 8e-3, "differ": 0.0} if whole else {"rel": 4e-5, "max": 4e-3, "differ": 0.0}
    return {"rel": 4e-6 if whole else 2e-6, "max": 1e-4, "differ": 0.0}


# ----------------------------------------------------------------- exact ----


def exact(case, seed):
    """run()'s answer in 64 bits.  Where the cache is fp16, its rows are rounded to fp16: they are stored results."""
    return _EXACT[case["kind"]](case, seed)


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope(x, first):
    """Rotates [..., token, d] at positions first, first + 1, ..., with the frequencies in fp32 as the model defines them."""
    d = x.shape[-1]
    power = [np.float32(THETA ** float(np.float32(2 * i) / np.float32(d))) for i in range(d // 2)]
    frequency = torch.tensor([np.float32(1.0) / p for p in power], device=x.device, dtype=torch.float32)
    position = torch.arange(first, first + x.shape[-2], device=x.device, dtype=torch.float32)
    angle = (position[:, None] * frequency[None, :]).to(x)  # the angle is an fp32 product
    c, s = angle.cos(), angle.sin()
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, keys, values, first):
    """Causal attention of q [head][token][d] at positions first .. over [kv_head][key][d]."""
    group, d = q.shape[0] // keys.shape[0], q.shape[-1]
    out = torch.empty_like(q)
    key = torch.arange(keys.shape[1], device=q.device)
    for b in range(0, q.shape[1], 1024):
        rows = slice(b, min(b + 1024, q.shape[1]))
        position = torch.arange(first + rows.start, first + rows.stop, device=q.device)
        hidden_keys = key[None, :] > position[:, None]
        for h in range(q.shape[0]):
            scores = (q[h, rows] @ keys[h // group].T.contiguous()) / math.sqrt(d)
            scores.masked_fill_(hidden_keys, -math.inf)
            out[h, rows] = torch.softmax(scores, -1) @ values[h // group]
    return out


def _heads(x, d):
    return x.reshape(x.shape[0], -1, d).transpose(0, 1)


def _layer_rows(w, x, first, keys, values, dtype):
    """A layer over rows x [token][hidden] at positions first ..; keys, values [kv_head][position][d] get their rows."""
    d = w["q_norm"].shape[0]
    n = _norm(x, w["input_norm"])
    q = _rope(_norm(_heads(n @ w["q_proj"].T, d), w["q_norm"]), first)
    k = _rope(_norm(_heads(n @ w["k_proj"].T, d), w["k_norm"]), first)
    end = first + x.shape[0]
    keys[:, first:end] = k.to(dtype).double()
    values[:, first:end] = _heads(n @ w["v_proj"].T, d).to(dtype).double()
    attention = _attend(q, keys[:, :end], values[:, :end], first)
    x = x + attention.transpose(0, 1).reshape(x.shape[0], -1) @ w["o_proj"].T
    n = _norm(x, w["post_attention_norm"])
    return x + (torch.nn.functional.silu(n @ w["gate_proj"].T) * (n @ w["up_proj"].T)) @ w["down_proj"].T


def _doubles(layer):
    return {n: t.double() for n, t in layer.items()}


def _exact_layer_step(case, seed):
    g = _generator(seed)
    hidden, _, _, _, d, _ = SHAPES[case["model"]]
    dtype, position = _kv(case)[1], case["position"]
    w = _doubles(_layer(g, case["model"]))
    keys, values = (torch.cat([t.double(), t.new_zeros((HEADS[1], 1, d)).double()], 1)
                    for t in _cache_rows(g, position, d, dtype))
    out = _layer_rows(w, _normal(g, (1, hidden)).double(), position, keys, values, dtype)
    return {"out": out[0], "cache": _page_views(keys, values, position + 1), "error": None}


def _exact_attention(case, seed):
    g = _generator(seed)
    d, tokens = case["head_dim"], case["tokens"]
    keys, values = _cache_rows(g, tokens, d, _kv(case)[1])
    q = _normal(g, (HEADS[0] * d,)).double().reshape(HEADS[0], 1, d)
    return {"out": _attend(q, keys.double(), values.double(), tokens - 1).reshape(-1)}


def _exact_head(case, seed):
    g = _generator(seed)
    w = _weight(g, case["rows"], case["hidden"]).double()
    x = _normal(g, (case["hidden"],), 3.0).double()
    logits = w @ _norm(x, _gain(g, case["hidden"]).double())
    return {"logits": logits, "token": logits.argmax().reshape(1).int()}


def _exact_projection(case, seed):
    g = _generator(seed)
    w = _weight(g, case["rows"], case["cols"]).double()
    y = _normal(g, (case["batch"], case["cols"])).double() @ w.T
    return {"y": y + _normal(g, (case["batch"], case["rows"])).double() if case["residual"] else y}


def _exact_layer_prompt(case, seed):
    g = _generator(seed)
    hidden, _, _, _, d, _ = SHAPES[case["model"]]
    w, tokens = _doubles(_layer(g, case["model"])), case["tokens"]
    dtype = _kv(case)[1]
    keys = torch.zeros((HEADS[1], tokens, d), device=DEVICE, dtype=torch.float64)
    values = torch.zeros_like(keys)
    _cache_rows(g, 0, d, dtype)
    out = _layer_rows(w, _normal(g, (tokens, hidden)).double(), 0, keys, values, dtype)
    return {"out": out, "cache": _page_views(keys, values, tokens)}


def _exact_prompt_attention(case, seed):
    g = _generator(seed)
    d, start, tokens = case["head_dim"], case["start"], case["tokens"]
    dtype = _kv(case)[1]
    keys, values = (torch.cat([t.double(), torch.zeros((HEADS[1], tokens, d), device=DEVICE, dtype=torch.float64)], 1)
                    for t in _cache_rows(g, start, d, dtype))
    qkv = _heads(_normal(g, (tokens, (HEADS[0] + 2 * HEADS[1]) * d), 0.6).double(), d)
    q_norm, k_norm = _gain(g, d).double(), _gain(g, d).double()
    q = _rope(_norm(qkv[: HEADS[0]], q_norm), start)
    keys[:, start:] = _rope(_norm(qkv[HEADS[0]: HEADS[0] + HEADS[1]], k_norm), start).to(dtype).double()
    values[:, start:] = qkv[HEADS[0] + HEADS[1]:].to(dtype).double()
    rows = lambda t: t.transpose(0, 1).reshape(tokens, -1)  # noqa: E731
    return {"query": rows(q), "out": rows(_attend(q, keys, values, start)),
            "cache": _page_views(keys, values, start + tokens)}


class _Exact64:
    """A whole model in 64 bits."""

    def __init__(self, case, seed):
        tensors = {n: t.double() for n, t in _model_weights(case, seed)}
        _, self.layers, _, _, self.d, _ = SHAPES[case["model"]]
        self.embed, self.final = tensors["model.embed_tokens.weight"], tensors["model.norm.weight"]
        self.dtype = _kv(case)[1]
        names = {"input_norm": "input_layernorm", "post_attention_norm": "post_attention_layernorm",
                 "q_norm": "self_attn.q_norm", "k_norm": "self_attn.k_norm", "gate_proj": "mlp.gate_proj",
                 "up_proj": "mlp.up_proj", "down_proj": "mlp.down_proj"}
        names.update({n + "_proj": "self_attn.%s_proj" % n for n in "qkvo"})
        self.w = [{n: tensors["model.layers.%d.%s.weight" % (i, f)] for n, f in names.items()}
                  for i in range(self.layers)]

    def generate(self, prompt, count):
        """(logits of the last step, the prompt and the `count` tokens after it)."""
        shape = (self.layers, HEADS[1], len(prompt) + count, self.d)
        keys = torch.zeros(shape, device=DEVICE, dtype=torch.float64)
        values = torch.zeros_like(keys)
        ids, done = [int(t) for t in prompt], 0
        for _ in range(count):
            x = self.embed[torch.tensor(ids[done:], device=DEVICE)]
            for i in range(self.layers):
                x = _layer_rows(self.w[i], x, done, keys[i], values[i], self.dtype)
            done = len(ids)
            logits = self.embed @ _norm(x[-1], self.final)
            ids.append(int(logits.argmax()))
        return logits.cpu().numpy(), np.array(ids, np.int32)


def _exact_model(case, seed):
    logits, ids = _Exact64(case, seed).generate(_prompts(case, seed)[0], case["steps"] + 1)
    return {"logits": logits, "tokens": ids[case["prompt"]:]}


def _exact_batch(case, seed):
    model, total = _Exact64(case, seed), case["prompt"] + case["steps"] + 1
    rows = [model.generate(p, total - len(p)) for p in _prompts(case, seed)]
    return {"logits": np.stack([r[0] for r in rows]), "tokens": np.stack([r[1] for r in rows])}


_EXACT = {"layer_step": _exact_layer_step, "attention": _exact_attention, "head": _exact_head,
          "projection": _exact_projection, "layer_prompt": _exact_layer_prompt,
          "prompt_attention": _exact_prompt_attention, "model": _exact_model, "batch": _exact_batch}
