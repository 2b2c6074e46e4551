"""The work that serving with this package consists of, as timed cases.

Four kinds of case, all through public entry points:

  attention      the attention of one serving step: `layers` calls of the
                 attn_fn over their own K/V caches with one step's metadata
                 (the first call of the step builds the decode plan).  Decode
                 steps replay a HIP graph, as the engine's do; steps that hold
                 prompt tokens run eagerly, as the engine's do.
  mlp            `layers` INT4 g128 MLPs with RMSNorm and residual
                 (Qwen2MLP), graph-replayed at decode batch sizes and called
                 eagerly at prompt sizes.
  model_decode   one decode step of the Qwen2.5-0.5B architecture in INT4 from
                 host-side sequences to logits and greedy tokens (DecodeGraphs).
  model_prefill  one prompt step of the same model, eager: inputs staged from
                 host-side sequences, forward, logits of each prompt's last row.

Context lengths and prompt lengths belong to the case (its `lengths` number);
weights, caches, queries and tokens come from the seed.
"""

from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from nanoserve_amd.attention import get_attention_backend
from nanoserve_amd.block_manager import BlockSpaceManager
from nanoserve_amd.capture import graph_capture
from nanoserve_amd.engine import ModelRunner
from nanoserve_amd.kv_cache import PagedKVCache
from nanoserve_amd.model import Qwen2Config, Qwen2ForCausalLM, Qwen2MLP, RMSNorm
from nanoserve_amd.quant import quantize_model
from nanoserve_amd.rotary import RotaryEmbedding
from nanoserve_amd.scheduling import SamplingParams, Sequence
from nanoserve_amd.workloads import metadata_for

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
GROUP = 128

# (query heads, KV heads, head size): the 0.5B model's, the larger-GQA
# benchmark's, and group sizes 1, 8 and 16 that the attention tests run.
HEADS = ((14, 2, 64), (28, 4, 128), (16, 2, 128), (8, 8, 64), (32, 2, 64))


def listed():
    return [
        # Decode, 8 short contexts (64..512 tokens): a lightly loaded server.
        # Per call a few us: launches and memory latency.
        _attention("decode_small", "uniform", 8, 64, 512, layers=24, lengths=1),
        # Decode at serving load, 32 contexts around 1K: the headline benchmark.
        _attention("decode_serving", "lognormal", 32, 16, 8192, median=1024, sigma=0.8, layers=24, lengths=2),
        # Long-context decode of a larger GQA model in bf16: the KV stream.
        _attention("decode_long", "lognormal", 64, 128, 32768, median=4096, sigma=1.0, layers=2, lengths=3,
                   heads=(28, 4, 128), dtype="bf16"),
        # A continuous-batching step: 28 decode rows and four 512-token prompt
        # chunks on top of up to 2K of context.
        _attention("mixed", "lognormal", 28, 16, 8192, median=1024, sigma=0.8, layers=24, lengths=4,
                   chunks=4, chunk=512, chunk_context=2048),
        # The late chunk of a long prompt: 2048 new tokens (the engine's
        # default step budget) behind ~12K of context.
        _attention("prefill_chunk", "uniform", 0, 1, 1, layers=4, lengths=5, chunks=1, chunk=2048,
                   chunk_context=14001),
        # Whole prompts of a larger GQA model in bf16, ragged, 8K-token budget.
        _attention("prefill_prompts", "uniform", 0, 1, 1, layers=1, lengths=6, chunks=2, chunk=4097,
                   chunk_context=0, heads=(28, 4, 128), dtype="bf16"),
        # The 0.5B model's MLPs at a full decode batch.
        _mlp("mlp_decode", 896, 4864, 32, layers=24),
        # A wide model's MLPs (the 28 x 128-wide residual of the larger GQA
        # heads, 4x inside) at a decode batch: the weight stream.
        _mlp("mlp_wide_decode", 3584, 14336, 16, layers=4, dtype="bf16"),
        # ... and at an engine step's prompt budget, a few rows short of it.
        _mlp("mlp_wide_prefill", 3584, 14336, 2000, layers=1, dtype="bf16"),
        # One interactive request.
        _decode("model_decode_one", 1, 300, 300, lengths=7),
        # A full decode batch.
        _decode("model_decode_batch", 32, 100, 900, lengths=8),
        # A prompt step at the default 2048-token budget, three ragged prompts.
        {"name": "model_prefill", "kind": "model_prefill", "prompts": 3, "tokens": 2048, "lengths": 9},
    ]


def _attention(name, law, batch, lo, hi, median=0, sigma=0.0, layers=1, lengths=0, chunks=0, chunk=0,
               chunk_context=0, heads=(14, 2, 64), dtype="fp16", block=16, index="int64"):
    c = {"kind": "attention", "law": law, "batch": batch, "lo": lo, "hi": hi, "median": median, "sigma": sigma,
         "layers": layers, "lengths": lengths, "chunks": chunks, "chunk": chunk, "chunk_context": chunk_context,
         "hq": heads[0], "hkv": heads[1], "dim": heads[2], "dtype": dtype, "block": block, "index": index}
    return c if name is None else {"name": name, **c}


def _mlp(name, hidden, inter, tokens, layers, dtype="fp16"):
    c = {"kind": "mlp", "hidden": hidden, "inter": inter, "tokens": tokens, "layers": layers, "dtype": dtype}
    return c if name is None else {"name": name, **c}


def _decode(name, batch, lo, hi, lengths):
    c = {"kind": "model_decode", "batch": batch, "lo": lo, "hi": hi, "lengths": lengths}
    return c if name is None else {"name": name, **c}


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "mixed", "prefill", "mlp", "mlp", "model_decode", "model_prefill"])
    lengths = rng.randrange(1 << 20)
    heads = rng.choice(HEADS)
    more = {"heads": heads, "dtype": rng.choice(["fp16", "bf16"]), "block": rng.choice([16, 16, 32]),
            "index": rng.choice(["int32", "int64"]), "lengths": lengths}
    per_token = 4 * heads[1] * heads[2]  # K and V bytes of a token
    if kind == "decode":
        batch = _log_int(rng, 1, 64)
        # at most the K/V of the largest listed decode step
        median = _log_int(rng, 48, max(64, min(6000, int(3e8 / (per_token * batch)))))
        layers = max(1, min(24, int(4e8 / (per_token * batch * median))))
        return _attention(None, "lognormal", batch, 1, 6 * median, median=median, sigma=rng.choice([0.3, 0.8]),
                          layers=layers, **more)
    if kind == "mixed":
        chunk = _log_int(rng, 17, 700)
        return _attention(None, "lognormal", _log_int(rng, 1, 48), 1, 6000, median=_log_int(rng, 64, 1500),
                          sigma=0.8, layers=4, chunks=rng.choice([1, 2, 3, 4]), chunk=chunk,
                          chunk_context=rng.choice([0, _log_int(rng, 16, 3000)]), **more)
    if kind == "prefill":
        chunks = rng.choice([1, 1, 2, 4])
        return _attention(None, "uniform", 0, 1, 1, layers=2, chunks=chunks,
                          chunk=_log_int(rng, 100, 4000 // chunks),
                          chunk_context=rng.choice([0, _log_int(rng, 16, 8000 // chunks)]), **more)
    if kind == "mlp":
        hidden, inter = rng.choice([(896, 4864), (896, 4864), (1536, 8960), (2048, 8192), (3584, 14336)])
        tokens = _log_int(rng, 1, 4000 if hidden < 2000 else 1999)
        layers = max(1, min(24, int(1.6e11 / (6 * hidden * inter * max(64, tokens)))))
        return _mlp(None, hidden, inter, tokens, layers, more["dtype"])
    if kind == "model_decode":
        return _decode(None, _log_int(rng, 1, 64), 16, _log_int(rng, 64, 1900), lengths)
    return {"kind": "model_prefill", "prompts": rng.choice([1, 2, 4, 8]), "tokens": _log_int(rng, 64, 2048),
            "lengths": lengths}


def _uses_graph(case):
    if case["kind"] == "attention":
        return case["chunks"] == 0
    return case["kind"] == "model_decode" or (case["kind"] == "mlp" and case["tokens"] <= 64)


# ---------------------------------------------------------------- lengths

def _step_lengths(case):
    """(context lengths including this step, query lengths) of an attention step."""
    rng = np.random.default_rng(case["lengths"])
    n = case["batch"]
    if case["law"] == "uniform":
        lens = rng.integers(case["lo"], case["hi"], size=n, endpoint=True)
    else:
        lens = np.clip(rng.lognormal(np.log(case["median"]), case["sigma"], n).astype(int), case["lo"], case["hi"])
    lens, q = [int(v) for v in lens], [1] * n
    for _ in range(case["chunks"]):
        ctx = int(rng.integers(0, case["chunk_context"], endpoint=True))
        # ragged prompts: up to a fifth shorter than the largest
        ql = case["chunk"] if case["chunk_context"] else int(rng.integers(case["chunk"] * 4 // 5, case["chunk"],
                                                                         endpoint=True))
        lens.append(ctx + ql)
        q.append(ql)
    return lens, q


def _model_lengths(case):
    rng = np.random.default_rng(case["lengths"])
    if case["kind"] == "model_decode":
        return [int(v) for v in rng.integers(case["lo"], max(case["lo"], case["hi"]), size=case["batch"],
                                             endpoint=True)]
    cuts = sorted(int(v) for v in rng.choice(np.arange(1, case["tokens"]), size=case["prompts"] - 1, replace=False))
    return [b - a for a, b in zip([0] + cuts, cuts + [case["tokens"]])]


# ---------------------------------------------------------------- inputs

def _randn(shape, g, dtype, std=1.0):
    return (torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std).to(dtype)


def _attention_inputs(case, seed):
    """(queries, k caches, v caches) per layer and the step's shuffled block tables."""
    lens, q = _step_lengths(case)
    need = [max(1, -(-n // case["block"])) for n in lens]
    pool = math.ceil(1.25 * sum(need))
    perm = np.random.default_rng(seed).permutation(pool).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n])
        at += n
    g = torch.Generator(device=DEV).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    layers = []
    for _ in range(case["layers"]):
        shape = (pool, case["block"], case["hkv"], case["dim"])
        layers.append((_randn((sum(q), case["hq"], case["dim"]), g, dtype), _randn(shape, g, dtype),
                       _randn(shape, g, dtype)))
    return lens, q, tables, layers


def _mlp_weights(case, seed):
    """Per layer (gate, up, down, norm weight), then the residual stream's rows."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    h, n = case["hidden"], case["inter"]
    layers = [(_randn((n, h), g, dtype, 0.02), _randn((n, h), g, dtype, 0.02), _randn((h, n), g, dtype, 0.02),
               1 + _randn((h,), g, dtype, 0.1)) for _ in range(case["layers"])]
    return layers, [_randn((case["tokens"], h), g, dtype) for _ in range(case["layers"])]


def _model_weights(seed):
    """The 0.5B architecture's parameters by name, N(0, 0.02) as the package initialises them."""
    cfg = Qwen2Config()
    g = torch.Generator(device=DEV).manual_seed(seed)
    h, n, kv = cfg.hidden_size, cfg.intermediate_size, cfg.num_key_value_heads * cfg.head_dim
    shapes = {"model.embed_tokens.weight": (cfg.vocab_size, h), "model.norm.weight": (h,)}
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        for name, rows in (("q", h), ("k", kv), ("v", kv)):
            shapes[f"{p}self_attn.{name}_proj.weight"] = (rows, h)
            shapes[f"{p}self_attn.{name}_proj.bias"] = (rows,)
        shapes[p + "self_attn.o_proj.weight"] = (h, h)
        shapes[p + "mlp.gate_proj.weight"] = shapes[p + "mlp.up_proj.weight"] = (n, h)
        shapes[p + "mlp.down_proj.weight"] = (h, n)
        shapes[p + "input_layernorm.weight"] = shapes[p + "post_attention_layernorm.weight"] = (h,)
    return cfg, {name: 1 + _randn(shape, g, torch.float16, 0.1) if name.endswith("norm.weight")
                 else _randn(shape, g, torch.float16, 0.02) for name, shape in shapes.items()}


def _model_state(case, seed):
    lens = _model_lengths(case)
    rng = np.random.default_rng(seed)
    cfg, weights = _model_weights(seed)
    need = [-(-n // 16) for n in lens]
    blocks = math.ceil(1.25 * sum(need))
    tokens = [rng.integers(0, cfg.vocab_size, n).tolist() for n in lens]
    perm = rng.permutation(blocks).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n])
        at += n
    g = torch.Generator(device=DEV).manual_seed(seed + 1)
    shape = (blocks, 16, cfg.num_key_value_heads, cfg.head_dim)
    # What earlier steps left in the cache (a prompt step overwrites its rows).
    caches = [(_randn(shape, g, torch.float16), _randn(shape, g, torch.float16))
              for _ in range(cfg.num_hidden_layers)]
    return cfg, weights, lens, tokens, tables, blocks, caches


def _captured(fn):
    """A graph of fn (warmed up on the capture stream first) and its outputs."""
    s = _stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with graph_capture(graph, stream=s):
        out = fn()
    return graph, out


_capture_stream = []


def _stream():
    if not _capture_stream:
        _capture_stream.append(torch.cuda.Stream())
    return _capture_stream[0]


def prepare(case, seed):
    with torch.inference_mode():
        return {"attention": _prepare_attention, "mlp": _prepare_mlp, "model_decode": _prepare_decode,
                "model_prefill": _prepare_prefill}[case["kind"]](case, seed)


def _prepare_attention(case, seed):
    attn, _ = get_attention_backend("auto")
    lens, q, tables, layers = _attention_inputs(case, seed)
    md = metadata_for(lens, q, tables, case["block"], DEV, {"int32": torch.int32, "int64": torch.int64}[case["index"]])
    scale = case["dim"] ** -0.5

    def step():
        step_md = dataclasses.replace(md, decode_plan=None)  # a step's metadata is new
        return [attn(x, k, v, step_md, scale) for x, k, v in layers]

    if _uses_graph(case):
        # A captured step knows no host-side lengths: they change under it.
        md = dataclasses.replace(md, query_lens_cpu=None, seq_lens_cpu=None, query_start_loc_cpu=None)
        graph, out = _captured(step)
        return {"graph": graph, "out": out, "keep": (md, layers)}
    return {"step": step}


def _prepare_mlp(case, seed):
    weights, xs = _mlp_weights(case, seed)
    cfg = Qwen2Config(hidden_size=case["hidden"], intermediate_size=case["inter"], num_hidden_layers=1)
    dtype = DTYPES[case["dtype"]]
    layers = []
    for gate, up, down, norm_w in weights:
        with torch.device(DEV):
            mlp, norm = Qwen2MLP(cfg).to(dtype), RMSNorm(case["hidden"], 1e-6).to(dtype)
        for lin, w in ((mlp.gate_proj, gate), (mlp.up_proj, up), (mlp.down_proj, down)):
            lin.weight.data.copy_(w)
        norm.weight.data.copy_(norm_w)
        quantize_model(mlp, GROUP)
        mlp.fuse()
        layers.append((mlp, norm))

    def step():
        return [mlp(x, residual=x, norm=norm) for (mlp, norm), x in zip(layers, xs)]

    if _uses_graph(case):
        graph, out = _captured(step)
        return {"graph": graph, "out": out, "keep": (layers, xs)}
    return {"step": step}


def _model_runner(case, seed, use_graphs):
    cfg, weights, lens, tokens, tables, blocks, caches = _model_state(case, seed)
    with torch.device(DEV):
        model = Qwen2ForCausalLM(cfg, max_position=8).half()
    model.model.rotary = RotaryEmbedding(cfg.head_dim, 2048, base=cfg.rope_theta)
    for name, p in model.named_parameters():
        p.data.copy_(weights[name])
    quantize_model(model, GROUP, skip=("lm_head",))
    model.fuse_projections().eval().requires_grad_(False)
    kv = PagedKVCache(blocks, 16, cfg.num_hidden_layers, cfg.num_key_value_heads, cfg.head_dim, torch.float16, DEV)
    for i, (k, v) in enumerate(caches):
        kv.k_cache[i].copy_(k)
        kv.v_cache[i].copy_(v)
    runner = ModelRunner(model, kv, BlockSpaceManager(16, blocks, watermark=0.0), DEV, use_graphs=use_graphs,
                         max_model_len=2048, graph_batch_sizes=(case.get("batch", 1),))
    seqs = []
    for i, (toks, table) in enumerate(zip(tokens, tables)):
        s = Sequence(i, toks, SamplingParams(max_new_tokens=16, ignore_eos=True))
        s.block_table = table
        s.num_computed_tokens = len(toks) - 1 if use_graphs else 0
        seqs.append(s)
    return runner, seqs, lens


def _prepare_decode(case, seed):
    runner, seqs, _ = _model_runner(case, seed, True)
    cached = [(k.clone(), v.clone()) for k, v in zip(runner.kv_cache.k_cache, runner.kv_cache.v_cache)]
    runner.graphs.capture_all()  # set-up, before serving
    # Capturing runs the model on padding rows only (no slot is written).
    for (k, v), kc, vc in zip(cached, runner.kv_cache.k_cache, runner.kv_cache.v_cache):
        kc.copy_(k)
        vc.copy_(v)
    return {"graphs": runner.graphs, "scheduled": [(s, 1) for s in seqs], "keep": runner}


def _prepare_prefill(case, seed):
    runner, seqs, lens = _model_runner(case, seed, False)
    return {"runner": runner, "scheduled": list(zip(seqs, lens))}


@torch.inference_mode()
def run(state):
    if "step" in state:
        return state["step"]()
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if "graphs" in state:
        # One engine step: fill, replay, read the greedy tokens back.
        graphs = state["graphs"]
        launch = graphs.launch(state["scheduled"])
        graphs.tokens(launch)
        return graphs.last_logits
    runner = state["runner"]
    ids, positions, md, rows, _ = runner.build_inputs(state["scheduled"])
    hidden = runner.model(ids, positions, runner.kv_cache, md, runner.attn_fn)
    return runner.model.compute_logits(hidden, rows)


# ---------------------------------------------------------------- what a pass needs

def _pairs(lens, q):
    """(query, key) pairs of a causal step."""
    return sum(n * (L - n) + n * (n + 1) // 2 for L, n in zip(lens, q))


def _int4_bytes(n, k):
    return n * k // 2 + n * (k // GROUP) * 5


def work(case):
    if case["kind"] == "attention":
        lens, q = _step_lengths(case)
        size = torch.tensor([], dtype=DTYPES[case["dtype"]]).element_size()
        row = case["dim"] * size
        nbytes = 2 * sum(lens) * case["hkv"] * row + 2 * sum(q) * case["hq"] * row
        return {"bytes": case["layers"] * nbytes,
                "flops": case["layers"] * 4 * case["hq"] * case["dim"] * _pairs(lens, q)}
    if case["kind"] == "mlp":
        h, n, t = case["hidden"], case["inter"], case["tokens"]
        nbytes = _int4_bytes(2 * n, h) + _int4_bytes(h, n) + 2 * 2 * t * h
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * 6 * t * h * n}
    cfg = Qwen2Config()
    lens = _model_lengths(case)
    q = [1] * len(lens) if case["kind"] == "model_decode" else lens
    h, n, layers = cfg.hidden_size, cfg.intermediate_size, cfg.num_hidden_layers
    qkv = h + 2 * cfg.num_key_value_heads * cfg.head_dim
    per_layer = _int4_bytes(qkv, h) + _int4_bytes(h, h) + _int4_bytes(2 * n, h) + _int4_bytes(h, n)
    kv = 2 * cfg.num_key_value_heads * cfg.head_dim * 2
    head = cfg.vocab_size * h
    nbytes = layers * (per_layer + kv * sum(lens)) + 2 * head + 2 * len(lens) * cfg.vocab_size
    flops = layers * (2 * sum(q) * h * (qkv + h + 3 * n) + 4 * h * _pairs(lens, q)) + 2 * len(lens) * head
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance from 64 bits that was measured (2.7e-4 for an
    attention or MLP call in fp16, 2.1e-3 / 4.5e-3 in bf16, 4.8e-3 for 24 layers
    of fp16): two correct roundings of the same value differ by both their errors."""
    if case["kind"] == "attention":
        return {"rel": 0.0011 if case["dtype"] == "fp16" else 0.0085}
    if case["kind"] == "mlp":
        return {"rel": 0.0011 if case["dtype"] == "fp16" else 0.018}
    return {"rel": 0.02}


# ---------------------------------------------------------------- 64 bits

def _attend64(q, keys, values, scale):
    """Causal attention of the last len(q) of len(keys) positions; [n, Hq, D], [L, Hkv, D]."""
    n, hq, d = q.shape
    L, hkv, _ = keys.shape
    q = q.double().view(n, hkv, hq // hkv, d).permute(1, 2, 0, 3).contiguous()  # [Hkv, G, n, D]
    kt = keys.double().permute(1, 2, 0).contiguous()   # [Hkv, D, L]
    vt = values.double().permute(1, 0, 2).contiguous()  # [Hkv, L, D]
    out = torch.empty_like(q)
    rows = max(1, min(n, int(2e8 / (L * hq // hkv))))
    at = torch.arange(L, device=DEV)
    for h in range(hkv):
        for i in range(0, n, rows):
            x = q[h, :, i:i + rows]
            s = torch.matmul(x, kt[h]) * scale
            last = torch.arange(i, i + x.shape[1], device=DEV) + (L - n)
            s.masked_fill_(at[None, None, :] > last[None, :, None], float("-inf"))
            out[h, :, i:i + rows] = torch.matmul(torch.softmax(s, -1), vt[h])
    return out.permute(2, 0, 1, 3).reshape(n, hq, d)


def _rows_of(cache, table, length):
    idx = torch.tensor(table, device=DEV)
    return cache.index_select(0, idx).reshape(-1, *cache.shape[2:])[:length]


def _int4_64(w):
    """The 64-bit weight that INT4 g128 codes of w stand for, rounded to w's dtype as the format defines."""
    n, k = w.shape
    wg = w.float().reshape(n, k // GROUP, GROUP)
    lo, hi = wg.amin(2, keepdim=True), wg.amax(2, keepdim=True)
    scale = ((hi - lo) / 15.0).clamp(min=1e-8)
    zero = (-lo / scale).round().clamp(0, 15)
    code = ((wg / scale).round() + zero).clamp(0, 15)
    return ((code - zero) * scale).to(w.dtype).double().reshape(n, k)


def _norm64(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _silu64(x):
    return x * torch.sigmoid(x)


@torch.inference_mode()
def exact(case, seed):
    if case["kind"] == "attention":
        lens, q, tables, layers = _attention_inputs(case, seed)
        outs = []
        for x, k, v in layers:
            parts, at = [], 0
            for L, n, t in zip(lens, q, tables):
                parts.append(_attend64(x[at:at + n], _rows_of(k, t, L), _rows_of(v, t, L), case["dim"] ** -0.5))
                at += n
            outs.append(torch.cat(parts))
        return outs
    if case["kind"] == "mlp":
        weights, xs = _mlp_weights(case, seed)
        outs = []
        for (gate, up, down, norm_w), x in zip(weights, xs):
            x = x.double()
            y = _norm64(x, norm_w)
            act = _silu64(y @ _int4_64(gate).t()) * (y @ _int4_64(up).t())
            outs.append(x + act @ _int4_64(down).t())
        return outs
    return _model64(case, seed)


def _model64(case, seed):
    cfg, w, lens, tokens, tables, _, caches = _model_state(case, seed)
    hq, hkv, d = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    q = [1] * len(lens) if case["kind"] == "model_decode" else lens
    ids = torch.tensor([t for toks, n in zip(tokens, q) for t in toks[len(toks) - n:]], device=DEV)
    pos = torch.cat([torch.arange(L - n, L, device=DEV) for L, n in zip(lens, q)])
    # The rotary table is float32 rounded to the model dtype, as the model defines it.
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, d, 2, dtype=torch.float32) / d))
    freqs = torch.outer(pos.cpu().float(), inv)
    emb = torch.cat((freqs, freqs), -1)
    cos, sin = (t.half().double().to(DEV)[:, None, :] for t in (emb.cos(), emb.sin()))

    def rotate(x):
        return x * cos + torch.cat((-x[..., d // 2:], x[..., :d // 2]), -1) * sin

    hidden = w["model.embed_tokens.weight"][ids].double()
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        x = _norm64(hidden, w[p + "input_layernorm.weight"])
        xq, xk, xv = (x @ _int4_64(w[f"{p}self_attn.{n}_proj.weight"]).t()
                      + w[f"{p}self_attn.{n}_proj.bias"].double() for n in "qkv")
        xq, xk, xv = rotate(xq.view(-1, hq, d)), rotate(xk.view(-1, hkv, d)), xv.view(-1, hkv, d)
        parts, at = [], 0
        for L, n, t in zip(lens, q, tables):
            keys, values = (torch.cat((_rows_of(c, t, L - n).double(), new[at:at + n]))
                            for c, new in zip(caches[i], (xk, xv)))
            parts.append(_attend64(xq[at:at + n], keys, values, d ** -0.5))
            at += n
        hidden = hidden + torch.cat(parts).view(-1, hq * d) @ _int4_64(w[p + "self_attn.o_proj.weight"]).t()
        x = _norm64(hidden, w[p + "post_attention_layernorm.weight"])
        act = _silu64(x @ _int4_64(w[p + "mlp.gate_proj.weight"]).t()) * (x @ _int4_64(w[p + "mlp.up_proj.weight"]).t())
        hidden = hidden + act @ _int4_64(w[p + "mlp.down_proj.weight"]).t()
    rows = torch.tensor(np.cumsum(q) - 1, device=DEV)
    hidden = _norm64(hidden[rows], w["model.norm.weight"])
    return hidden @ w["model.embed_tokens.weight"].double().t()
