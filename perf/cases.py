"""The measured workloads: what a serving program has this package do.

Every case is one pass through public entry points, with the inputs, plans and
buffers that such a program holds before the call:

* ``decode``: one layer's attention of a pure-decode step
  (``MI355XAttentionBackend.forward`` on the step's plan); with ``store`` the
  layer also writes the step's new K/V rows (``forward_with_kv_store``);
* ``prefill``: one layer's attention of a prefill step, over new tokens that
  follow cached ones (a prefix hit, or the earlier chunks of a long prompt);
* ``mixed``: one layer's attention of a chunked-prefill step, prefill chunks
  and decodes in one batch;
* ``layer``: what a decoder layer launches besides its GEMMs and attention:
  residual add + RMSNorm, q/k norm + RoPE + KV store, residual add + RMSNorm,
  SiLU-and-mul;
* ``graph``: the same launches and the decode attention between them, captured
  once in a HIP graph and replayed, as a decode step of few sequences runs.

A step's plan is built once for all of a model's layers, so it is part of what
``prepare`` hands over; lengths are drawn per case (``lengths`` seeds them),
values and page permutations from the seed.  Contexts, head counts, hidden
sizes and batch sizes are those of the repository's benchmark configurations
(Qwen3-0.6B, 8B and 32B layers and their tensor-parallel shards, page 16,
head_dim 128) and of the steps between them.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from my_vllm_amd import ops
from my_vllm_amd.attention_backend import MI355XAttentionBackend
from my_vllm_amd.contract import CommonAttentionMetadata
from my_vllm_amd.custom_op import CustomOpConfig
from my_vllm_amd.layers import RMSNorm, RotaryEmbedding, SiluAndMul

PAGE = 16
DIM = 128
EPS = 1e-6
ROPE_BASE = 1000000.0
MAX_POSITION = 40960
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
# (hidden size, MLP width, query heads, KV heads) of the three model sizes.
MODELS = ((1024, 3072, 16, 8), (4096, 12288, 32, 8), (5120, 25600, 64, 8))
# Whole layers, then tensor-parallel shards of them.
HEADS = ((16, 8), (32, 8), (64, 8), (16, 4), (32, 4), (16, 2), (8, 1))
# A drawn attention case moves or computes no more than the largest listed one.
MAX_KV_BYTES = 5.0e9
MAX_STORE_BYTES = 4.0e8
MAX_PREFILL_FLOPS = 3.4e11


def listed():
    return [
        # A decode step of a few interactive users, in a captured graph: the
        # smallest launches, where latency and launch gaps are the time.
        {"name": "graph_layer_8seq", "kind": "graph", "dtype": "bf16", "hq": 16, "hkv": 8, "hidden": 1024,
         "inter": 3072, "batch": 8, "ctx_lo": 256, "ctx_hi": 1024, "lengths": 11},
        # One user with a long document.
        {"name": "decode_1seq_30k", "kind": "decode", "dtype": "bf16", "hq": 32, "hkv": 8, "batch": 1,
         "ctx_lo": 30001, "ctx_hi": 30001, "store": False, "lengths": 0},
        # The headline decode batch, new rows stored by the same call.
        {"name": "decode_64seq_2k_store", "kind": "decode", "dtype": "bf16", "hq": 16, "hkv": 8, "batch": 64,
         "ctx_lo": 128, "ctx_hi": 2048, "store": True, "lengths": 1},
        # Half of an 8B layer's heads (tensor parallelism over two GPUs), fp16.
        {"name": "decode_37seq_6k_shard_fp16", "kind": "decode", "dtype": "fp16", "hq": 16, "hkv": 4, "batch": 37,
         "ctx_lo": 300, "ctx_hi": 6000, "store": False, "lengths": 5},
        # Long-context decode at the 32B shape: the largest K/V read.
        {"name": "decode_56seq_32k", "kind": "decode", "dtype": "bf16", "hq": 64, "hkv": 8, "batch": 56,
         "ctx_lo": 8192, "ctx_hi": 32768, "store": False, "lengths": 4},
        # One short prompt without a cached prefix (time to first token).
        {"name": "prefill_1seq_333", "kind": "prefill", "dtype": "bf16", "hq": 16, "hkv": 8, "seqs": 1,
         "q_lo": 333, "q_hi": 333, "prefix_lo": 0, "prefix_hi": 0, "lengths": 0},
        # A 512-token chunk late in a long prompt.
        {"name": "prefill_chunk_512_over_7k", "kind": "prefill", "dtype": "bf16", "hq": 32, "hkv": 8, "seqs": 1,
         "q_lo": 512, "q_hi": 512, "prefix_lo": 7168, "prefix_hi": 7168, "lengths": 0},
        # The benchmark's batch of prompts with cached prefixes.
        {"name": "prefill_16seq_prefix", "kind": "prefill", "dtype": "bf16", "hq": 32, "hkv": 8, "seqs": 16,
         "q_lo": 64, "q_hi": 2048, "prefix_lo": 0, "prefix_hi": 1024, "lengths": 2},
        # A lightly loaded server: one prompt's chunk beside twenty decodes.
        {"name": "mixed_300_20dec_fp16", "kind": "mixed", "dtype": "fp16", "hq": 32, "hkv": 8, "seqs": 1,
         "q_lo": 300, "q_hi": 300, "prefix_lo": 0, "prefix_hi": 2048, "decodes": 20, "ctx_lo": 128, "ctx_hi": 4096,
         "lengths": 7},
        # The benchmark's chunked-prefill step at a token budget of 8192.
        {"name": "mixed_budget_8192", "kind": "mixed", "dtype": "bf16", "hq": 32, "hkv": 8, "seqs": 4,
         "q_lo": 512, "q_hi": 2048, "prefix_lo": 0, "prefix_hi": 8192, "decodes": 256, "ctx_lo": 512,
         "ctx_hi": 8192, "lengths": 3},
        # The launches around the GEMMs of an 8B layer: a decode step of 61
        # sequences, and a prefill step.
        {"name": "layer_61tok", "kind": "layer", "dtype": "bf16", "hq": 32, "hkv": 8, "hidden": 4096,
         "inter": 12288, "tokens": 61},
        {"name": "layer_4099tok", "kind": "layer", "dtype": "bf16", "hq": 32, "hkv": 8, "hidden": 4096,
         "inter": 12288, "tokens": 4099},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choices(("decode", "prefill", "mixed", "layer", "graph"), (35, 25, 15, 15, 10))[0]
    case = {"kind": kind, "dtype": rng.choice(("bf16", "bf16", "fp16"))}
    if kind in ("layer", "graph"):
        hidden, inter, hq, hkv = rng.choice(MODELS)
        case.update(hidden=hidden, inter=inter, hq=hq, hkv=hkv)
        if kind == "layer":
            case["tokens"] = _log_int(rng, 1, 6000 if hidden < 5120 else 4000)
            return case
    else:
        case["hq"], case["hkv"] = rng.choice(HEADS)
    case["lengths"] = rng.randrange(1 << 16)
    row = 2 * case["hkv"] * DIM * 2  # K/V bytes of one token
    if kind in ("decode", "graph"):
        case["batch"] = _log_int(rng, 1, 256 if kind == "decode" else 64)
        hi = _log_int(rng, 32, 32768 if kind == "decode" else 4096)
        limit = MAX_KV_BYTES if kind == "decode" else MAX_STORE_BYTES
        if kind == "decode":
            case["store"] = rng.random() < 0.3 and case["batch"] * hi * row <= MAX_STORE_BYTES
        hi = max(32, min(hi, int(limit / row / case["batch"])))
        case["ctx_hi"] = hi
        case["ctx_lo"] = max(1, hi // rng.choice((1, 2, 4, 16)))
        return case
    case["seqs"] = _log_int(rng, 1, 24) if kind == "prefill" else rng.randint(1, 4)
    case["q_hi"] = _log_int(rng, 16, 6000 if kind == "prefill" else 2048)
    case["q_lo"] = max(1, case["q_hi"] // rng.choice((1, 2, 8, 32)))
    case["prefix_hi"] = rng.choice((0, _log_int(rng, 16, 8192), _log_int(rng, 16, 16384)))
    case["prefix_lo"] = rng.choice((0, case["prefix_hi"]))
    if kind == "mixed":
        case["decodes"] = _log_int(rng, 1, 256)
        case["ctx_hi"] = min(_log_int(rng, 64, 16384), int(0.8 * MAX_KV_BYTES / row / case["decodes"]))
        case["ctx_lo"] = max(1, case["ctx_hi"] // rng.choice((1, 2, 16)))
    while work(case)["flops"] > MAX_PREFILL_FLOPS * (1 if kind == "prefill" else 1.1):
        if kind == "mixed" and case["decodes"] > 1 and case["q_hi"] < 64:
            case["decodes"] //= 2
        case["q_hi"] = max(1, case["q_hi"] * 3 // 4)
        case["q_lo"] = min(case["q_lo"], case["q_hi"])
        case["prefix_hi"] = case["prefix_hi"] * 7 // 8
        case["prefix_lo"] = min(case["prefix_lo"], case["prefix_hi"])
    return case


def _lengths(case):
    """(query lengths, context lengths, prefill sequences) of an attention case."""
    rng = np.random.default_rng(case["lengths"])

    def uniform(lo, hi, n):
        return [int(x) for x in rng.integers(lo, hi + 1, size=n)]

    if case["kind"] in ("decode", "graph"):
        ctx = uniform(case["ctx_lo"], case["ctx_hi"], case["batch"])
        return [1] * len(ctx), ctx, 0
    q = uniform(case["q_lo"], case["q_hi"], case["seqs"])
    # Cached prefixes are whole pages; a chunk may follow any token.
    step = PAGE if case["kind"] == "prefill" else 1
    prefix = [step * x for x in uniform(case["prefix_lo"] // step, case["prefix_hi"] // step, case["seqs"])]
    kv = [a + b for a, b in zip(q, prefix)]
    if case["kind"] == "mixed":
        kv += uniform(case["ctx_lo"], case["ctx_hi"], case["decodes"])
        q += [1] * case["decodes"]
    return q, kv, case["seqs"]


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _normal(gen, dtype, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)


def _attention_state(case, gen):
    """The paged batch of one step: queries, new K/V rows, caches, metadata."""
    dtype = DTYPES[case["dtype"]]
    hq, hkv = case["hq"], case["hkv"]
    q_len, kv_len, prefills = _lengths(case)
    counts = [(n + PAGE - 1) // PAGE for n in kv_len]
    pages = sum(counts)
    order = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32)
    width = max(counts)
    used = torch.arange(width, device="cuda")[None, :] < torch.tensor(counts, device="cuda")[:, None]
    table = torch.full((len(counts), width), -1, dtype=torch.int32, device="cuda")
    table[used] = order
    positions = np.concatenate([np.arange(n - q, n) for q, n in zip(q_len, kv_len)])
    rows = np.repeat(np.arange(len(q_len)), q_len)
    positions = torch.from_numpy(positions).to("cuda")
    rows = torch.from_numpy(rows).to("cuda")
    slots = table[rows, positions // PAGE] * PAGE + (positions % PAGE).to(torch.int32)
    starts = np.concatenate(([0], np.cumsum(q_len))).astype(np.int32)
    total = int(starts[-1])
    common = CommonAttentionMetadata(
        num_prefill_seqs=prefills, num_decode_seqs=len(q_len) - prefills,
        num_prefill_tokens=int(sum(q_len[:prefills])), num_decode_tokens=int(sum(q_len[prefills:])),
        query_start_loc=torch.from_numpy(starts).to("cuda"),
        seq_lens=torch.tensor(kv_len, dtype=torch.int32, device="cuda"),
        slot_mapping=slots.contiguous(), block_tables=table, max_q_len=max(q_len), max_kv_len=max(kv_len),
        block_counts=tuple(counts), num_kv_blocks=pages, num_prefill_kv_blocks=sum(counts[:prefills]),
        trusted=True,
    )
    return {
        "case": case, "common": common, "positions": positions,
        "q": _normal(gen, dtype, total, hq, DIM),
        "k": _normal(gen, dtype, total, hkv, DIM),
        "v": _normal(gen, dtype, total, hkv, DIM),
        "k_cache": _normal(gen, dtype, pages, PAGE, hkv, DIM),
        "v_cache": _normal(gen, dtype, pages, PAGE, hkv, DIM),
    }


def _layer_inputs(case, gen, tokens):
    """A layer's hidden states, residual and GEMM outputs, and its weights."""
    dtype = DTYPES[case["dtype"]]
    heads = case["hq"] + 2 * case["hkv"]
    return {
        "hidden": _normal(gen, dtype, tokens, case["hidden"]),
        "residual": _normal(gen, dtype, tokens, case["hidden"]),
        "attn_proj": _normal(gen, dtype, tokens, case["hidden"]),
        "gate_up": _normal(gen, dtype, tokens, 2 * case["inter"]),
        "qkv": _normal(gen, dtype, tokens, heads, DIM),
        "w1": 1 + 0.1 * _normal(gen, dtype, case["hidden"]),
        "w2": 1 + 0.1 * _normal(gen, dtype, case["hidden"]),
        "wq": 1 + 0.1 * _normal(gen, dtype, DIM),
        "wk": 1 + 0.1 * _normal(gen, dtype, DIM),
    }


def _layer_cache(case, gen, tokens):
    """A cache half again as large as the step, its rows at random slots, and
    the tokens' positions."""
    dtype = DTYPES[case["dtype"]]
    pages = (3 * tokens // 2 + PAGE - 1) // PAGE + 1
    return {
        "positions": torch.randint(0, MAX_POSITION, (tokens,), generator=gen, device="cuda"),
        "slots": torch.randperm(pages * PAGE, generator=gen, device="cuda")[:tokens].to(torch.int32),
        "k_cache": _normal(gen, dtype, pages, PAGE, case["hkv"], DIM),
        "v_cache": _normal(gen, dtype, pages, PAGE, case["hkv"], DIM),
    }


def _layer_modules(case, state):
    dtype = DTYPES[case["dtype"]]
    config = CustomOpConfig(platform="cuda", dtype=dtype)

    def norm(width, weight):
        module = RMSNorm(width, EPS, config).to(device="cuda", dtype=dtype).requires_grad_(False)
        module.weight.copy_(weight)
        return module

    state["norm1"] = norm(case["hidden"], state["w1"])
    state["norm2"] = norm(case["hidden"], state["w2"])
    state["q_norm"] = norm(DIM, state["wq"])
    state["k_norm"] = norm(DIM, state["wk"])
    state["rope"] = RotaryEmbedding(DIM, DIM, MAX_POSITION, ROPE_BASE, config).to("cuda")
    state["act"] = SiluAndMul(config)
    state["rotated"] = torch.empty_like(state["qkv"])


def _run_layer(s, attention):
    """The layer's launches in order; ``attention`` runs between them."""
    hq, hkv = s["case"]["hq"], s["case"]["hkv"]
    h1, res = s["norm1"](s["hidden"], s["residual"])
    q, k, v = s["qkv"].split((hq, hkv, hkv), dim=1)
    # Into buffers of its own, so that a pass can be repeated on one state.
    q_out, k_out, _ = s["rotated"].split((hq, hkv, hkv), dim=1)
    ops.qk_norm_rope_store(s["positions"], q, k, s["rope"].cos_sin_cache, s["q_norm"].weight, s["k_norm"].weight,
                           EPS, v, s["k_cache"], s["v_cache"], s["slots"], q_out, k_out)
    outputs = [h1, q_out, k_out, s["k_cache"], s["v_cache"]]
    if attention is not None:
        outputs.append(attention(q_out))
    h2, res2 = s["norm2"](s["attn_proj"], res)
    outputs += [res, h2, res2, s["act"](s["gate_up"])]
    return outputs


def _capture(case, s):
    backend = s["backend"]
    common = s["common"]
    plan = backend.build_plan(common)
    batch, width = common.block_tables.shape
    graph_state = backend.create_full_decode_graph_state(batch, batch * width, torch.device("cuda"))
    backend.plan_full_decode_graph(graph_state, plan)
    empty = s["qkv"].new_empty((0, case["hkv"], DIM))

    def attention(q):
        return backend.forward(q, empty, empty, s["k_cache"], s["v_cache"], plan)

    backend.activate_full_decode_graph(graph_state)
    try:
        _run_layer(s, attention)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            s["outputs"] = _run_layer(s, attention)
        torch.cuda.synchronize()
    finally:
        backend.deactivate_full_decode_graph()
    s["graph"], s["graph_state"] = graph, graph_state


def prepare(case, seed):
    gen = _generator(seed)
    if case["kind"] == "layer":
        state = {"case": case, **_layer_inputs(case, gen, case["tokens"]), **_layer_cache(case, gen, case["tokens"])}
        _layer_modules(case, state)
        return state
    state = _attention_state(case, gen)
    state["backend"] = MI355XAttentionBackend(case["hq"], case["hkv"], DIM, PAGE, DTYPES[case["dtype"]])
    if case["kind"] == "graph":
        state.update(_layer_inputs(case, gen, case["batch"]))
        state["slots"] = state["common"].slot_mapping
        _layer_modules(case, state)
        _capture(case, state)
        return state
    state["plan"] = state["backend"].build_plan(state["common"])
    return state


def run(state):
    kind = state["case"]["kind"]
    if kind == "layer":
        return _run_layer(state, None)
    if kind == "graph":
        state["graph"].replay()
        return state["outputs"]
    s = state
    if s["case"].get("store"):
        out = s["backend"].forward_with_kv_store(s["q"], s["k"], s["v"], s["k_cache"], s["v_cache"],
                                                 s["common"].slot_mapping, s["plan"])
        return [out, s["k_cache"], s["v_cache"]]
    return s["backend"].forward(s["q"], s["k"], s["v"], s["k_cache"], s["v_cache"], s["plan"])


def work(case):
    """Each K/V row, query, output and page id once; two products per visible
    (query, key) pair and head.  Layer launches: each input and output once."""
    heads = case["hq"] + 2 * case["hkv"]
    moved = flops = 0
    if case["kind"] in ("layer", "graph"):
        tokens = case["tokens"] if case["kind"] == "layer" else case["batch"]
        # The second norm's residual comes from the first.
        norms = 2 * 4 * case["hidden"]
        rope = (2 * heads + case["hkv"]) * DIM
        moved += 2 * tokens * (norms + rope + 3 * case["inter"]) + tokens * (4 * DIM + 12)
        flops += tokens * (10 * case["hidden"] + 10 * heads * DIM + 6 * case["inter"])
        if case["kind"] == "layer":
            return {"bytes": moved, "flops": flops}
    q_len, kv_len, _ = _lengths(case)
    pairs = sum(q * (n - q) + q * (q + 1) // 2 for q, n in zip(q_len, kv_len))
    moved += sum(kv_len) * 2 * case["hkv"] * DIM * 2 + 2 * sum(q_len) * case["hq"] * DIM * 2
    moved += sum((n + PAGE - 1) // PAGE for n in kv_len) * 4
    if case.get("store"):
        moved += sum(q_len) * 4 * case["hkv"] * DIM * 2
    flops += 4 * DIM * case["hq"] * pairs
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # Rounding of the stored results, and of the probabilities (attention) or
    # the normed rows (layer) before their product, to the storage type.
    # Against float64, bf16 results measured up to 3.5e-3 (2-norm) and 6e-2
    # (largest), fp16 results up to 4.5e-4 and 7e-3: about four times that.
    if case["dtype"] == "bf16":
        return {"rel": 1.2e-2, "max": 0.25}
    return {"rel": 1.8e-3, "max": 0.03}


def _exact_attention(case, common, q, k_cache, v_cache):
    """Causal attention over the paged cache, in float64."""
    hkv, group = case["hkv"], case["hq"] // case["hkv"]
    q_len, kv_len, _ = _lengths(case)
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    first = 0
    for s, (n, kv) in enumerate(zip(q_len, kv_len)):
        pages = common.block_tables[s, : (kv + PAGE - 1) // PAGE].long()
        k = k_cache[pages].reshape(-1, hkv, DIM)[:kv].double().permute(1, 2, 0).contiguous()
        v = v_cache[pages].reshape(-1, hkv, DIM)[:kv].double().permute(1, 0, 2).contiguous()
        for a in range(0, n, 256):
            b = min(a + 256, n)
            rows = q[first + a : first + b].double().reshape(b - a, hkv, group, DIM)
            rows = rows.permute(1, 2, 0, 3).reshape(hkv, group * (b - a), DIM).contiguous()
            scores = torch.matmul(rows, k).view(hkv, group, b - a, kv) / math.sqrt(DIM)
            last = torch.arange(kv - n + a, kv - n + b, device="cuda")
            scores.masked_fill_(torch.arange(kv, device="cuda")[None, :] > last[:, None], -math.inf)
            part = torch.matmul(torch.softmax(scores, -1).view(hkv, -1, kv), v)
            out[first + a : first + b] = part.view(hkv, group, b - a, DIM).permute(2, 0, 1, 3).reshape(b - a, -1, DIM)
        first += n
    return out


def _exact_rms(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _exact_layer(case, s, attention):
    hq, hkv = case["hq"], case["hkv"]
    # The layer's fp32 table is an input: its values as they are.
    freq = 1.0 / torch.pow(ROPE_BASE, torch.arange(0, DIM, 2, dtype=torch.float32) / DIM)
    angle = torch.outer(torch.arange(MAX_POSITION, dtype=torch.float32), freq)
    cos = angle.cos().to("cuda")[s["positions"]].double()[:, None, :]
    sin = angle.sin().to("cuda")[s["positions"]].double()[:, None, :]

    def rotate(x):
        x1, x2 = x[..., : DIM // 2], x[..., DIM // 2 :]
        return torch.cat((x1 * cos - x2 * sin, x2 * cos + x1 * sin), -1)

    res = s["hidden"].double() + s["residual"].double()
    q, k, v = s["qkv"].double().split((hq, hkv, hkv), dim=1)
    q, k = rotate(_exact_rms(q, s["wq"])), rotate(_exact_rms(k, s["wk"]))
    k_cache, v_cache = s["k_cache"].double(), s["v_cache"].double()
    k_cache.view(-1, hkv, DIM)[s["slots"].long()] = k
    v_cache.view(-1, hkv, DIM)[s["slots"].long()] = v
    outputs = [_exact_rms(res, s["w1"]), q, k, k_cache, v_cache]
    if attention:
        outputs.append(_exact_attention(case, s["common"], q, k_cache, v_cache))
    res2 = res + s["attn_proj"].double()
    gate, up = s["gate_up"].double().chunk(2, -1)
    outputs += [res, _exact_rms(res2, s["w2"]), res2, gate * torch.sigmoid(gate) * up]
    return outputs


def exact(case, seed):
    gen = _generator(seed)
    if case["kind"] == "layer":
        state = {**_layer_inputs(case, gen, case["tokens"]), **_layer_cache(case, gen, case["tokens"])}
        return _exact_layer(case, state, False)
    s = _attention_state(case, gen)
    if case["kind"] == "graph":
        s.update(_layer_inputs(case, gen, case["batch"]))
        s["slots"] = s["common"].slot_mapping
        return _exact_layer(case, s, True)
    if case.get("store"):
        for cache, new in ((s["k_cache"], s["k"]), (s["v_cache"], s["v"])):
            cache.view(-1, case["hkv"], DIM)[s["common"].slot_mapping.long()] = new
    out = _exact_attention(case, s["common"], s["q"], s["k_cache"], s["v_cache"])
    if case.get("store"):
        return [out, s["k_cache"].double(), s["v_cache"].double()]
    return out
