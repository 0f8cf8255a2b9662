"""The work a user of this framework has it do, as cases that can be timed.

Whole calls run the repository's model, Llama-3.2-1B's geometry at full size
(16 layers, vocabulary 128256, seeded random weights), through `Model`:

  prompt     one prompt through `Model.prefill`, to its last position's logits
  reply      tokens of a running conversation through `Model.decode`, one call
             each, over the positions already cached, to the last one's logits

A change of rounding in one layer travels through the sixteen: two correct
bf16 prompts (other chunk lengths, so other summation orders) have logits 2.4
to 2.9 % apart, two fp16 ones 0.33 %. So whole prompts that run as matrix
products are compared on the fp16 build; shorter ones and decoding, whose
order of summation is fixed, on either.

Layer calls run parts of a layer through the kernel entry points
(include/lcr_kernels.h) as a host that keeps its own model loop calls them:

  attention  the attention half of a layer for a chunk of a prompt: embedding
             rows, input norm, q/k/v projection with RoPE and the cache append,
             causal attention over the cache, output projection joined to the
             residual, and the norm after it
  mlp        the other half: embedding rows, norm, gate/up with SwiGLU, down
             joined to the residual, and the next norm
  cached     one decoded token's attention over the cached positions
  sample     the next id from fp32 logits by temperature, top-k and top-p
"""

import importlib
import json
import math
import os
import shutil
import tempfile
from pathlib import Path

import numpy as np
import torch

lcr = importlib.import_module("llama-cuda-runtime_amd")

DEVICE = "cuda:0"
ELEM = {"bf16": torch.bfloat16, "fp16": torch.float16}
HIDDEN, FFN, VOCAB, LAYERS = 2048, 8192, 128256, 16
KV_HEADS = 8
ROWS = 4096  # embedding rows behind the layer calls' token ids
PAGE = 16
EPS = 1e-5
COMPUTE_UNITS = 256


def listed():
    return [
        # the first message of a chat: 27 tokens, the prompt length that the
        # reference's own benchmark is quoted on; what the user waits for first
        {"name": "prompt_27", "kind": "prompt", "tokens": 27, "paged": False, "dtype": "bf16"},
        # a pasted page of text on the fp16 build with a paged cache
        {"name": "prompt_700_fp16", "kind": "prompt", "tokens": 700, "paged": True, "dtype": "fp16"},
        # a paragraph of answer behind 128 cached positions: batch-1 decoding,
        # the headline workload, at its context
        {"name": "reply_64", "kind": "reply", "context": 128, "steps": 64, "paged": False, "dtype": "bf16"},
        # a layer over a system prompt with a short question
        {"name": "attention_128", "kind": "attention", "tokens": 128, "start": 0, "head_dim": 64, "paged": False,
         "dtype": "bf16"},
        # a layer over the longest prompt that runs as one chunk
        {"name": "attention_2048", "kind": "attention", "tokens": 2048, "start": 0, "head_dim": 64, "paged": False,
         "dtype": "bf16"},
        # the last, ragged chunk of a long document, over what the earlier
        # chunks left in a paged cache (fp16 build)
        {"name": "attention_chunk_fp16", "kind": "attention", "tokens": 500, "start": 6144, "head_dim": 64,
         "paged": True, "dtype": "fp16"},
        # a chat message of ordinary, odd length on the fp16 build
        {"name": "mlp_77_fp16", "kind": "mlp", "tokens": 77, "dtype": "fp16"},
        # the benchmark's two prefill sizes
        {"name": "mlp_512", "kind": "mlp", "tokens": 512, "dtype": "bf16"},
        {"name": "mlp_2048", "kind": "mlp", "tokens": 2048, "dtype": "bf16"},
        # one token early in a conversation: the smallest call, all latency
        {"name": "cached_300", "kind": "cached", "positions": 300, "head_dim": 64, "paged": False, "dtype": "bf16"},
        # one token after a long document, paged
        {"name": "cached_8192", "kind": "cached", "positions": 8192, "head_dim": 64, "paged": True, "dtype": "bf16"},
        # the sampling settings of the sampled-generation benchmark
        {"name": "sample_top40", "kind": "sample", "vocab": VOCAB, "temperature": 0.8, "top_k": 40, "top_p": 0.95},
    ]


def _spread(rng, low, high):
    """A whole number from low to high, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "reply", "attention", "attention", "mlp", "mlp", "cached", "sample"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    paged = rng.random() < 0.4
    if kind == "prompt":
        tokens = _spread(rng, 2, 2048)
        return {"kind": kind, "tokens": tokens, "paged": paged, "dtype": dtype if tokens < 64 else "fp16"}
    if kind == "reply":
        return {"kind": kind, "context": _spread(rng, 16, 32768), "steps": _spread(rng, 4, 40), "paged": paged,
                "dtype": dtype}
    if kind == "attention":
        return {"kind": kind, "tokens": _spread(rng, 64, 2048), "start": rng.choice([0, 0, _spread(rng, 64, 4096)]),
                "head_dim": rng.choice([64, 64, 128]), "paged": paged, "dtype": dtype}
    if kind == "mlp":
        return {"kind": kind, "tokens": _spread(rng, 64, 2048), "dtype": dtype}
    if kind == "cached":
        return {"kind": kind, "positions": _spread(rng, 1, 32768), "head_dim": rng.choice([64, 64, 128]),
                "paged": paged, "dtype": dtype}
    return {"kind": kind, "vocab": rng.choice([VOCAB, _spread(rng, 4096, VOCAB)]),
            "temperature": round(rng.uniform(0.5, 1.2), 2), "top_k": rng.choice([0, 1, 40, 64, 100]),
            "top_p": rng.choice([1.0, 0.95, 0.9])}


# ---------------------------------------------------------------------------
# inputs


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(gen, shape, std, dtype):
    return (torch.randn(shape, device=DEVICE, generator=gen) * std).to(ELEM[dtype])


def _checkpoint(dtype):
    """The full-size model's directory, written once per machine and user:
    every state holds the same weights, as a server's model does."""
    home = Path(tempfile.gettempdir()) / f"llama_cases_{os.getuid()}_{dtype}_{lcr.WEIGHT_SEED}"
    if not (home / "config.json").exists():
        fresh = tempfile.mkdtemp(prefix="llama_cases_", dir=tempfile.gettempdir())
        lcr.write_synthetic_checkpoint(fresh, fp16=dtype == "fp16")
        try:
            os.rename(fresh, home)
        except OSError:  # another process was first
            shutil.rmtree(fresh, ignore_errors=True)
    return home


def _prepare_model(case, seed):
    """The model and the ids it is given; a reply's cached positions hold
    normal keys and values, as this model's own are distributed."""
    count = case["tokens"] if case["kind"] == "prompt" else case["steps"]
    context = case.get("context", 0)
    model = lcr.Model(_checkpoint(case["dtype"]), variant=case["dtype"], max_seq=context + count + 1,
                      paged=case["paged"], page_size=PAGE)
    if context:
        model.fill_kv_normal(seed, 1.0)
    return {"model": model, "ids": np.random.default_rng(seed).integers(0, VOCAB, count).astype(np.int32),
            "logits": torch.empty(VOCAB, device=DEVICE, dtype=torch.float32)}


def _heads(case):
    """Query heads: 32 of 64 or 16 of 128, always on eight kv heads."""
    return HIDDEN // case["head_dim"]


def _cache(gen, case, positions, filled):
    """A cache of `positions` positions of which the first `filled` hold
    normal values, and the view the kernels take. Pages lie in random order."""
    head_dim, dtype = case["head_dim"], case["dtype"]
    view = lcr.KvView()
    table = None
    if case["paged"]:
        pages = -(-positions // PAGE)
        shape = (pages, KV_HEADS, PAGE, head_dim)
        table = torch.randperm(pages, device=DEVICE, generator=gen).to(torch.int32)
        view.page_table = table.data_ptr()
        view.page_size, view.page_stride, view.head_stride = PAGE, KV_HEADS * PAGE * head_dim, PAGE * head_dim
    else:
        shape = (KV_HEADS, positions, head_dim)
        view.page_size, view.page_stride, view.head_stride = 0, 0, positions * head_dim
    cache = {}
    for name in ("keys", "values"):
        t = torch.zeros(shape, device=DEVICE, dtype=ELEM[dtype])
        past = _normal(gen, (KV_HEADS, filled, head_dim), 1.0, dtype)
        _write_positions(t, table, past)
        cache[name] = t
    view.keys, view.values = cache["keys"].data_ptr(), cache["values"].data_ptr()
    view.num_kv_heads, view.head_dim = KV_HEADS, head_dim
    cache.update(view=view, table=table)
    return cache


def _write_positions(pool, table, past):
    at = torch.arange(past.shape[1], device=DEVICE)
    if table is None:
        pool[:, : past.shape[1]] = past
    else:
        pool[table[at // PAGE].long(), :, at % PAGE] = past.transpose(0, 1)


def _read_positions(pool, table, count):
    """[kv_heads][count][head_dim] of a cache pool."""
    if table is None:
        return pool[:, :count]
    at = torch.arange(count, device=DEVICE)
    return pool[table[at // PAGE].long(), :, at % PAGE].transpose(0, 1)


def _inv_freq(head_dim):
    """Llama 3's rotation frequencies (rope_scaling of the configuration)."""
    cfg = lcr.LLAMA_3_2_1B_CONFIG
    s = cfg["rope_scaling"]
    f = 1.0 / cfg["rope_theta"] ** (np.arange(0, head_dim, 2, dtype=np.float64) / head_dim)
    wave = 2 * np.pi / f
    old = s["original_max_position_embeddings"]
    smooth = (old / wave - s["low_freq_factor"]) / (s["high_freq_factor"] - s["low_freq_factor"])
    mixed = (1 - smooth) * f / s["factor"] + smooth * f
    f = np.where(wave > old / s["low_freq_factor"], f / s["factor"],
                 np.where(wave < old / s["high_freq_factor"], f, mixed))
    return torch.from_numpy(f.astype(np.float32)).to(DEVICE)


def _layer_inputs(gen, case):
    """Token ids, the embedding they index, two norms' weights and the buffers
    that a layer's halves write."""
    T, dtype = case["tokens"], case["dtype"]
    elem = ELEM[dtype]
    return {
        "ids": torch.randint(0, ROWS, (T,), device=DEVICE, generator=gen, dtype=torch.int32),
        "embedding": _normal(gen, (ROWS, HIDDEN), 1.0, dtype),
        "norm_in": (1.0 + 0.1 * torch.randn(HIDDEN, device=DEVICE, generator=gen)).to(elem),
        "norm_out": (1.0 + 0.1 * torch.randn(HIDDEN, device=DEVICE, generator=gen)).to(elem),
        "x": torch.empty(T, HIDDEN, device=DEVICE, dtype=elem),
        "normed": torch.empty(T, HIDDEN, device=DEVICE, dtype=elem),
        "delta": torch.empty(T, HIDDEN, device=DEVICE, dtype=elem),
        "out": torch.empty(T, HIDDEN, device=DEVICE, dtype=elem),
    }


def _workspace(lib, T, shapes):
    """One workspace for all of a layer's projections, as a model keeps it."""
    size = max(lib.lcr_gemm_workspace_bytes(T, n, k) for n, k in shapes)
    return torch.empty(max(size, 256), device=DEVICE, dtype=torch.uint8)


def _prepare_attention(case, seed):
    gen, lib = _generator(seed), lcr.load_library(case["dtype"])
    T, hd, dtype = case["tokens"], case["head_dim"], case["dtype"]
    heads = _heads(case)
    rows = (heads + 2 * KV_HEADS) * hd
    state = _layer_inputs(gen, case)
    state["w_qkv"] = _normal(gen, (rows, HIDDEN), 0.02, dtype)
    state["w_o"] = _normal(gen, (HIDDEN, HIDDEN), 0.02, dtype)
    state["q"] = torch.empty(heads, T, hd, device=DEVICE, dtype=ELEM[dtype])
    state["mixed"] = torch.empty(T, HIDDEN, device=DEVICE, dtype=ELEM[dtype])
    state["workspace"] = _workspace(lib, T, [(rows, HIDDEN), (HIDDEN, HIDDEN)])
    positions = case["start"] + T
    state["cache"] = _cache(gen, case, positions, case["start"])
    state["inv_freq"] = _inv_freq(hd)
    state["rope"] = torch.empty(positions, hd, device=DEVICE, dtype=torch.float32)
    lcr.check(lib, lib.lcr_rope_table(state["rope"].data_ptr(), state["inv_freq"].data_ptr(), positions, hd, None))
    return state


def _prepare_mlp(case, seed):
    gen, lib = _generator(seed), lcr.load_library(case["dtype"])
    T, dtype = case["tokens"], case["dtype"]
    state = _layer_inputs(gen, case)
    state["w_gate_up"] = _normal(gen, (2 * FFN, HIDDEN), 0.02, dtype)
    state["w_down"] = _normal(gen, (HIDDEN, FFN), 0.02, dtype)
    state["act"] = torch.empty(T, FFN, device=DEVICE, dtype=ELEM[dtype])
    state["workspace"] = _workspace(lib, T, [(2 * FFN, HIDDEN), (HIDDEN, FFN)])
    return state


def _prepare_cached(case, seed):
    gen, lib = _generator(seed), lcr.load_library(case["dtype"])
    heads, hd = _heads(case), case["head_dim"]
    splits = lib.lcr_choose_attention_splits(KV_HEADS, case["positions"], COMPUTE_UNITS)
    floats = lib.lcr_decode_attention_scratch_floats(heads, hd, splits)
    return {
        "cache": _cache(gen, case, case["positions"], case["positions"]),
        "q": _normal(gen, (heads, hd), 1.0, case["dtype"]),
        "out": torch.empty(heads, hd, device=DEVICE, dtype=ELEM[case["dtype"]]),
        "splits": splits,
        "scratch": torch.empty(max(floats, 4), device=DEVICE, dtype=torch.float32),
    }


def _prepare_sample(case, seed):
    gen, lib = _generator(seed), lcr.load_library("bf16")
    return {
        "logits": 3.0 * torch.randn(case["vocab"], device=DEVICE, generator=gen),
        "uniform": lcr.philox_uniforms(seed, 1)[0],
        "id": torch.empty(1, device=DEVICE, dtype=torch.int32),
        "scratch": torch.empty(lib.lcr_sample_scratch_floats(case["vocab"], case["top_k"]), device=DEVICE),
    }


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("prompt", "reply"):
        state = _prepare_model(case, seed)
    else:
        state = {"attention": _prepare_attention, "mlp": _prepare_mlp, "cached": _prepare_cached,
                 "sample": _prepare_sample}[kind](case, seed)
        state["lib"] = lcr.load_library(case.get("dtype", "bf16"))
    state["case"] = case
    return state


# ---------------------------------------------------------------------------
# one pass


def _run_model(state):
    model = state["model"]
    if state["case"]["kind"] == "prompt":
        model.reset()
        logits = model.prefill(state["ids"])
    else:
        model.set_position(state["case"]["context"])
        for token in state["ids"]:
            logits = model.decode(token)
    # the model's own buffer holds the logits only until its next call
    out = state["logits"]
    lcr.check(model.lib, model.lib.lcr_memcpy_dtod(out.data_ptr(), logits, out.nbytes))
    return out


def _embed_and_norm(lib, s, T, stream):
    p = torch.Tensor.data_ptr
    lcr.check(lib, lib.lcr_embedding_lookup(p(s["x"]), p(s["embedding"]), p(s["ids"]), T, HIDDEN, stream))
    lcr.check(lib, lib.lcr_rmsnorm(p(s["normed"]), p(s["x"]), p(s["norm_in"]), T, HIDDEN, EPS, stream))


def _run_attention(s, stream):
    case, lib, p = s["case"], s["lib"], torch.Tensor.data_ptr
    T, start, hd, paged = case["tokens"], case["start"], case["head_dim"], int(case["paged"])
    heads, view = _heads(case), s["cache"]["view"]
    ws, size = p(s["workspace"]), s["workspace"].numel()
    _embed_and_norm(lib, s, T, stream)
    lcr.check(lib, lib.lcr_gemm_qkv_rope_ws(p(s["q"]), view, p(s["normed"]), p(s["w_qkv"]), p(s["rope"]), T, heads,
                                            HIDDEN, start, paged, ws, size, stream))
    lcr.check(lib, lib.lcr_prefill_attention(p(s["mixed"]), p(s["q"]), view, heads, heads // KV_HEADS, T, start,
                                             hd ** -0.5, paged, stream))
    lcr.check(lib, lib.lcr_gemm_residual_rmsnorm_ws(p(s["out"]), p(s["x"]), p(s["delta"]), p(s["mixed"]), p(s["w_o"]),
                                                    p(s["norm_out"]), T, HIDDEN, HIDDEN, EPS, ws, size, stream))
    return {"q": s["q"], "keys": s["cache"]["keys"], "values": s["cache"]["values"], "mixed": s["mixed"],
            "x": s["x"], "out": s["out"]}


def _run_mlp(s, stream):
    lib, p, T = s["lib"], torch.Tensor.data_ptr, s["case"]["tokens"]
    ws, size = p(s["workspace"]), s["workspace"].numel()
    _embed_and_norm(lib, s, T, stream)
    lcr.check(lib, lib.lcr_gemm_swiglu_ws(p(s["act"]), p(s["normed"]), p(s["w_gate_up"]), T, FFN, HIDDEN, ws, size,
                                          stream))
    lcr.check(lib, lib.lcr_gemm_residual_rmsnorm_ws(p(s["out"]), p(s["x"]), p(s["delta"]), p(s["act"]), p(s["w_down"]),
                                                    p(s["norm_out"]), T, HIDDEN, FFN, EPS, ws, size, stream))
    return {"act": s["act"], "x": s["x"], "out": s["out"]}


def _run_cached(s, stream):
    case, lib, p = s["case"], s["lib"], torch.Tensor.data_ptr
    heads = _heads(case)
    lcr.check(lib, lib.lcr_decode_attention(p(s["out"]), p(s["q"]), s["cache"]["view"], heads, heads // KV_HEADS,
                                            case["positions"], case["head_dim"] ** -0.5, int(case["paged"]),
                                            s["splits"], p(s["scratch"]), stream))
    return s["out"]


def _run_sample(s, stream):
    case, lib, p = s["case"], s["lib"], torch.Tensor.data_ptr
    lcr.check(lib, lib.lcr_sample(p(s["id"]), p(s["logits"]), case["vocab"], case["temperature"], case["top_k"],
                                  case["top_p"], s["uniform"], p(s["scratch"]), stream))
    return s["id"]


def run(state):
    kind = state["case"]["kind"]
    if kind in ("prompt", "reply"):
        return _run_model(state)
    stream = torch.cuda.current_stream().cuda_stream
    return {"attention": _run_attention, "mlp": _run_mlp, "cached": _run_cached, "sample": _run_sample}[kind](
        state, stream)


# ---------------------------------------------------------------------------
# what a pass cannot do without

LAYER_WEIGHTS = 3072 * HIDDEN + HIDDEN * HIDDEN + 3 * FFN * HIDDEN + 2 * HIDDEN
HEAD_WEIGHTS = VOCAB * HIDDEN + HIDDEN


def _attention_flops(heads, head_dim, tokens, start):
    """Scores and weighted values over the keys each position sees."""
    seen = tokens * start + tokens * (tokens + 1) // 2
    return 4.0 * heads * head_dim * seen


def work(case):
    kind = case["kind"]
    e = 2
    if kind in ("prompt", "reply"):
        kv = 2 * LAYERS * KV_HEADS * 64 * e  # cache bytes a position
        if kind == "prompt":
            T = case["tokens"]
            flops = 2.0 * LAYER_WEIGHTS * LAYERS * T + 2.0 * HEAD_WEIGHTS + LAYERS * _attention_flops(32, 64, T, 0)
            return {"bytes": e * (LAYERS * LAYER_WEIGHTS + HEAD_WEIGHTS + T * HIDDEN) + kv * T + 4 * VOCAB,
                    "flops": flops}
        n, c = case["steps"], case["context"]
        read = n * c + n * (n + 1) // 2
        flops = n * 2.0 * (LAYER_WEIGHTS * LAYERS + HEAD_WEIGHTS) + LAYERS * 4.0 * HIDDEN * read
        return {"bytes": n * e * (LAYERS * LAYER_WEIGHTS + HEAD_WEIGHTS + HIDDEN) + kv * read + n * 4 * VOCAB,
                "flops": flops}
    if kind in ("attention", "mlp"):
        T = case["tokens"]
        rows = e * T * HIDDEN  # one [tokens][hidden] tensor
        if kind == "mlp":
            weights = 3 * FFN * HIDDEN
            return {"bytes": e * weights + 3 * rows + e * T * FFN, "flops": 2.0 * weights * T}
        hd = case["head_dim"]
        weights = (HIDDEN + 2 * KV_HEADS * hd) * HIDDEN + HIDDEN * HIDDEN
        cache = 2 * e * KV_HEADS * hd * (case["start"] + T)
        return {"bytes": e * weights + 5 * rows + cache,
                "flops": 2.0 * weights * T + _attention_flops(_heads(case), hd, T, case["start"])}
    if kind == "cached":
        n, hd = case["positions"], case["head_dim"]
        return {"bytes": 2 * e * KV_HEADS * hd * n + 2 * e * HIDDEN, "flops": 4.0 * HIDDEN * n}
    return {"bytes": 4 * case["vocab"] + 4, "flops": 4.0 * case["vocab"]}


def tolerance(case):
    """Four times what two correct implementations of the same precision
    differ by, where that is measured (the whole calls: see the top); for the
    layer calls, whose outputs are 0.2 to 0.4 % (bf16) and 0.01 to 0.05 %
    (fp16) off their 64-bit values, a few times that."""
    kind, bf16 = case["kind"], case.get("dtype") == "bf16"
    if kind == "sample":
        return "exact"
    if kind in ("prompt", "reply"):
        return {"rel": 0.03 if bf16 else 0.014}
    return {"rel": 0.012 if bf16 else 0.0016}


# ---------------------------------------------------------------------------
# the same in 64 bits, without the framework


def _rms64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rotate64(x, inv_freq, start):
    """Half-split RoPE of [heads][tokens][head_dim]; the angle is the 32-bit
    product that the framework defines."""
    half = x.shape[-1] // 2
    at = torch.arange(start, start + x.shape[1], device=DEVICE, dtype=torch.float32)
    angle = (at[:, None] * inv_freq[None, :]).double()
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * angle.cos() - hi * angle.sin(), hi * angle.cos() + lo * angle.sin()], -1)


def _attend64(q, keys, values, start):
    """Causal attention of [heads][tokens][head_dim] queries at positions from
    `start` on, heads in groups on the kv heads; [tokens][heads * head_dim]."""
    heads, T, hd = q.shape
    group = heads // keys.shape[0]
    seen = torch.arange(keys.shape[1], device=DEVICE)[None, :] <= torch.arange(start, start + T, device=DEVICE)[:, None]
    out = torch.empty(T, heads * hd, device=DEVICE, dtype=torch.float64)
    for h in range(heads):
        scores = (q[h] @ keys[h // group].t()) * hd ** -0.5
        scores.masked_fill_(~seen, -math.inf)
        out[:, h * hd:(h + 1) * hd] = torch.softmax(scores, -1) @ values[h // group]
    return out


def _split_heads(x, heads, head_dim):
    return x.reshape(x.shape[0], heads, head_dim).transpose(0, 1)


def _attention_half64(x, norm_in, w_qkv, w_o, inv_freq, heads, head_dim, start=0, past=None):
    """(queries, keys, values of these tokens, mixed heads, new residual)."""
    kv = KV_HEADS * head_dim
    qkv = _rms64(x, norm_in) @ w_qkv.double().t()
    q = _rotate64(_split_heads(qkv[:, :heads * head_dim], heads, head_dim), inv_freq, start)
    k = _rotate64(_split_heads(qkv[:, heads * head_dim:heads * head_dim + kv], KV_HEADS, head_dim), inv_freq, start)
    v = _split_heads(qkv[:, heads * head_dim + kv:], KV_HEADS, head_dim)
    all_k, all_v = (k, v) if past is None else (torch.cat([past[0], k], 1), torch.cat([past[1], v], 1))
    mixed = _attend64(q, all_k, all_v, start)
    return q, k, v, mixed, x + mixed @ w_o.double().t()


def _mlp_half64(x, norm, gate, up, down):
    n = _rms64(x, norm)
    act = torch.nn.functional.silu(n @ gate.double().t()) * (n @ up.double().t())
    return act, x + act @ down.double().t()


def _checkpoint_tensors(dtype):
    """name -> a loader of that tensor to the GPU, from the safetensors file."""
    path = _checkpoint(dtype) / "model.safetensors"
    with open(path, "rb") as f:
        size = int.from_bytes(f.read(8), "little")
        header = json.loads(f.read(size))
    data = np.memmap(path, dtype=np.uint8, mode="r", offset=8 + size)

    def load(name):
        at, shape = header[name]["data_offsets"], header[name]["shape"]
        raw = torch.from_numpy(np.array(data[at[0]:at[1]]))
        return raw.view(ELEM[dtype]).reshape(shape).to(DEVICE)

    return load


def _exact_model(case, seed):
    state = _prepare_model(case, seed)
    load, inv_freq, start = _checkpoint_tensors(case["dtype"]), _inv_freq(64), case.get("context", 0)
    embedding = load("model.embed_tokens.weight")
    x = embedding[torch.from_numpy(state["ids"].astype(np.int64)).to(DEVICE)].double()
    state["model"].set_position(start)
    for i in range(LAYERS):
        p = f"model.layers.{i}."
        past = None
        if start:
            past = [torch.from_numpy(t.view(np.int16)).view(ELEM[case["dtype"]]).to(DEVICE).double()
                    for t in state["model"].kv_export(i, start, KV_HEADS, 64)]
        qkv = torch.cat([load(p + f"self_attn.{n}_proj.weight") for n in "qkv"])
        x = _attention_half64(x, load(p + "input_layernorm.weight"), qkv, load(p + "self_attn.o_proj.weight"),
                              inv_freq, 32, 64, start, past)[-1]
        x = _mlp_half64(x, load(p + "post_attention_layernorm.weight"), load(p + "mlp.gate_proj.weight"),
                        load(p + "mlp.up_proj.weight"), load(p + "mlp.down_proj.weight"))[1]
    return embedding.double() @ _rms64(x[-1], load("model.norm.weight"))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prompt", "reply"):
        return _exact_model(case, seed)
    if kind == "sample":
        return None
    s = prepare(case, seed)
    if kind == "cached":
        c = s["cache"]
        keys, values = (_read_positions(c[n], c["table"], case["positions"]).double() for n in ("keys", "values"))
        mixed = _attend64(s["q"][:, None].double(), keys, values, case["positions"] - 1)
        return mixed.reshape(_heads(case), case["head_dim"])
    x = s["embedding"][s["ids"].long()].double()
    if kind == "mlp":
        gate, up = s["w_gate_up"][:FFN], s["w_gate_up"][FFN:]
        act, x = _mlp_half64(x, s["norm_in"], gate, up, s["w_down"])
        return {"act": act, "x": x, "out": _rms64(x, s["norm_out"])}
    c, start = s["cache"], case["start"]
    past = [_read_positions(c[n], c["table"], start).double() for n in ("keys", "values")]
    q, k, v, mixed, x = _attention_half64(x, s["norm_in"], s["w_qkv"], s["w_o"], s["inv_freq"], _heads(case),
                                          case["head_dim"], start, past)
    pools = []
    for name, old, new in (("keys", past[0], k), ("values", past[1], v)):
        pool = torch.zeros(c[name].shape, device=DEVICE, dtype=torch.float64)
        _write_positions(pool, c["table"], torch.cat([old, new], 1))
        pools.append(pool)
    return {"q": q, "keys": pools[0], "values": pools[1], "mixed": mixed, "x": x, "out": _rms64(x, s["norm_out"])}
