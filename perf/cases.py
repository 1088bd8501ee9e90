"""Performance cases: the work that a program using this framework has it do.

Every case goes through an entry point that the engine itself calls: the paged
attention ops (decode and chunked prefill), the pointwise ops, the sampler, one
decoder layer (decode and prefill) and one whole decode step of a model.
``listed()`` holds one case of each kind of work at the sizes of the benchmark
and test configurations; ``draw`` spreads further cases over the same ranges.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path.cwd() / "tiny-vllm_amd"))

PAGE = 16
VOCAB = 151936
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
# Decoder widths of the benchmark configurations: hidden, FFN, query heads.
WIDTHS = {"0.6b": (1024, 3072, 16), "8b": (4096, 12288, 32), "32b": (5120, 25600, 64)}
KV_HEADS = 8
HEAD_DIM = 128
EPS = 1e-6
THETA = 1_000_000.0


# ---------------------------------------------------------------- the cases --

def listed():
    return [
        # One chat request early in its answer: the smallest call, where
        # latency and launches count.
        dict(name="decode_1x300", kind="decode", rows=1, low=300, high=300, heads=16,
             kv_heads=8, dim=128, dtype="bf16", cache="same", layout="head_major"),
        # The headline batch: 64 requests at 2048 tokens, 8B heads.
        dict(name="decode_64x2048", kind="decode", rows=64, low=2048, high=2048, heads=32,
             kv_heads=8, dim=128, dtype="bf16", cache="same", layout="token_major"),
        # Long contexts over the FP8 cache, 32B heads, ragged lengths.
        dict(name="decode_16x32k_fp8", kind="decode", rows=16, low=16384, high=32768, heads=64,
             kv_heads=8, dim=128, dtype="bf16", cache="fp8", layout="head_major"),
        # Models with 64-wide heads in fp16, a ragged batch.
        dict(name="decode_33x4k_dim64", kind="decode", rows=33, low=1, high=4096, heads=32,
             kv_heads=8, dim=64, dtype="fp16", cache="same", layout="token_major"),
        # Chunked prefill: the last 512-token chunks of four 2048-token prompts.
        dict(name="prefill_4x512_2048", kind="prefill", items=4, query=512, ragged=False,
             history=1536, heads=32, kv_heads=8, dim=128, dtype="bf16", cache="same",
             layout="token_major"),
        # Short fresh prompts of odd lengths arriving together.
        dict(name="prefill_7_short", kind="prefill", items=7, query=201, ragged=True, history=0,
             heads=16, kv_heads=8, dim=128, dtype="bf16", cache="same", layout="token_major"),
        # Chunks of a model with 256-wide heads.
        dict(name="prefill_2x256_dim256", kind="prefill", items=2, query=256, ragged=False,
             history=777, heads=16, kv_heads=8, dim=256, dtype="bf16", cache="same",
             layout="token_major"),
        # The pointwise ops of one prefill chunk step at 8B widths.
        dict(name="pointwise_2048", kind="pointwise", tokens=2048, width="8b", dtype="bf16"),
        # One sampling call of a served batch: greedy, top-k and top-p requests.
        dict(name="sample_64", kind="sample", rows=64, vocab=VOCAB, dtype="bf16"),
        # One decoder layer of the headline decode step.
        dict(name="layer_decode_64x2048", kind="layer", width="8b", rows=64, low=2048, high=2048,
             query=1, layout="token_major"),
        # One decoder layer of a 512-token prefill chunk with history.
        dict(name="layer_prefill_512", kind="layer", width="8b", rows=1, low=2048, high=2048,
             query=512, layout="token_major"),
        # A whole graph-replayed decode step: embedding, layers, head, sampler.
        dict(name="step_16", kind="step", width="0.6b", layers=4, rows=16, low=64, high=1024),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    cap = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= cap:
            return case


def _draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "pointwise", "sample",
                       "layer", "layer", "step"])
    width = rng.choice(list(WIDTHS))
    heads = rng.choice([8, 16, 32, 64])
    attn = dict(heads=heads, kv_heads=8, dim=rng.choice([128, 128, 128, 64, 256, 32]),
                dtype=rng.choice(["bf16", "bf16", "fp16"]), cache=rng.choice(["same", "same", "fp8"]),
                layout=rng.choice(["token_major", "head_major"]))
    if kind == "decode":
        high = _log(rng, 64, 32768)
        return dict(kind=kind, rows=_log(rng, 1, 128), low=rng.choice([1, max(1, high // 2), high]),
                    high=high, **attn)
    if kind == "prefill":
        return dict(kind=kind, items=rng.randint(1, 8), query=_log(rng, 2, 1024),
                    ragged=rng.random() < 0.5, history=rng.choice([0, _log(rng, 1, 16384)]), **attn)
    if kind == "pointwise":
        return dict(kind=kind, tokens=_log(rng, 1, 4096), width=width,
                    dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "sample":
        return dict(kind=kind, rows=_log(rng, 1, 128), vocab=rng.choice([VOCAB, _log(rng, 1000, VOCAB)]),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if kind == "layer":
        layout = rng.choice(["token_major", "head_major"])
        if rng.random() < 0.6:
            high = _log(rng, 64, 8192)
            return dict(kind=kind, width=width, rows=_log(rng, 1, 128), low=max(1, high // 2),
                        high=high, query=1, layout=layout)
        query = _log(rng, 16, 1024)
        return dict(kind=kind, width=width, rows=rng.randint(1, 4), low=query, high=query + 512,
                    query=query, layout=layout)
    high = _log(rng, 64, 2048)
    return dict(kind=kind, width="0.6b", layers=rng.randint(1, 5), rows=_log(rng, 1, 64),
                low=max(1, high // 4), high=high)


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


# --------------------------------------------------------- inputs from a seed --

def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed) * 7919 + 17)


def _lengths(case):
    """Context lengths of the rows, uniform in [low, high], one at the top: the
    same ones for every seed, so that the outputs' shapes are the case's own."""
    g = _gen(case["rows"] * 100003 + case["high"], "cpu")
    lengths = torch.randint(case["low"], case["high"] + 1, (case["rows"],), generator=g)
    lengths[int(torch.randint(0, case["rows"], (1,), generator=g))] = case["high"]
    return lengths.tolist()


def _tables(contexts, seed):
    """Pages of each context drawn from a shuffled pool: (pool pages, tables)."""
    pages = [-(-n // PAGE) for n in contexts]
    pool = sum(pages) + 7
    order = torch.randperm(pool, generator=_gen(seed + 1, "cpu"))
    tables, at = [], 0
    for p in pages:
        tables.append(order[at:at + p])
        at += p
    return pool, tables


def _items(case):
    """(query lengths, context lengths) of a prefill call, the same for every seed."""
    n, q = case["items"], case["query"]
    if case["ragged"]:
        g = _gen(n * 100003 + q, "cpu")
        queries = torch.randint(max(2, q // 8), q + 1, (n,), generator=g).tolist()
        queries[-1] = q
    else:
        queries = [q] * n
    return queries, [x + case["history"] for x in queries]


def _slots(table, length, start=0):
    p = torch.arange(start, length)
    return table[p // PAGE] * PAGE + p % PAGE


def _attention_inputs(case, seed):
    """q, and the stored K and V rows [slots, kv_heads, dim] with their scales."""
    dt = DTYPES[case["dtype"]]
    if case["kind"] == "decode":
        queries, contexts = [1] * case["rows"], _lengths(case)
    else:
        queries, contexts = _items(case)
    pool, tables = _tables(contexts, seed)
    g = _gen(seed)
    q = torch.randn((sum(queries), case["heads"], case["dim"]), generator=g, device="cuda").to(dt)
    fp8 = case["cache"] == "fp8"
    ks, vs = (0.0625, 0.03125) if fp8 else (1.0, 1.0)
    kv = []
    for scale in (ks, vs):
        x = torch.randn((pool * PAGE, case["kv_heads"], case["dim"]), generator=g, device="cuda",
                        dtype=torch.float32 if dt == torch.float16 else dt)
        kv.append((x / scale).to(torch.float8_e4m3fn) if fp8 else x.to(dt))
    return queries, contexts, pool, tables, q, kv[0], kv[1], ks, vs


def _pointwise_inputs(case, seed):
    hidden, ffn, heads = WIDTHS[case["width"]]
    dt, n = DTYPES[case["dtype"]], case["tokens"]
    g = _gen(seed)

    def r(*shape, mean=0.0, std=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(dt)

    pool = -(-n // PAGE) + 5
    slots = torch.randperm(pool * PAGE, generator=_gen(seed, "cpu"))[:n].cuda()
    positions = torch.randint(0, 2048, (n,), generator=_gen(seed + 3, "cpu")).cuda()
    return dict(x=r(n, hidden), residual=r(n, hidden), weight=r(hidden, mean=1.0, std=0.02),
                qkv=r(n, (heads + 2 * KV_HEADS) * HEAD_DIM), q_weight=r(HEAD_DIM, mean=1.0, std=0.02),
                k_weight=r(HEAD_DIM, mean=1.0, std=0.02), gate_up=r(n, 2 * ffn), slots=slots,
                positions=positions, pool=pool, heads=heads)


def _layer_inputs(case, seed):
    """Weights, activations and KV contents of one decoder layer's step."""
    hidden, ffn, heads = WIDTHS[case["width"]]
    queries, after = [case["query"]] * case["rows"], _lengths(case)
    pool, tables = _tables(after, seed)
    g = _gen(seed)
    dt = torch.bfloat16

    def r(*shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=g, device="cuda", dtype=dt) * std + mean

    q_size, kv_size, tokens = heads * HEAD_DIM, KV_HEADS * HEAD_DIM, sum(queries)
    w = dict(qkv=r(q_size + 2 * kv_size, hidden, std=0.02), o=r(hidden, q_size, std=0.02),
             gate_up=r(2 * ffn, hidden, std=0.02), down=r(hidden, ffn, std=0.02),
             norm1=r(hidden, mean=1.0, std=0.02), norm2=r(hidden, mean=1.0, std=0.02),
             norm3=r(hidden, mean=1.0, std=0.02), q_norm=r(HEAD_DIM, mean=1.0, std=0.02),
             k_norm=r(HEAD_DIM, mean=1.0, std=0.02))
    x = dict(hidden=r(tokens, hidden), residual=r(tokens, hidden),
             key=r(pool * PAGE, KV_HEADS, HEAD_DIM), value=r(pool * PAGE, KV_HEADS, HEAD_DIM))
    positions = torch.cat([torch.arange(a - q, a) for q, a in zip(queries, after)])
    slots = torch.cat([_slots(t, a, a - q) for t, q, a in zip(tables, queries, after)])
    return queries, after, pool, tables, positions, slots, w, x


def _step_inputs(case, seed):
    """Weights, KV contents and rows of a whole decode step (tied embeddings)."""
    hidden, ffn, heads = WIDTHS[case["width"]]
    after = _lengths(case)
    pool, tables = _tables(after, seed)
    g = _gen(seed)
    dt = torch.bfloat16

    def r(*shape, std=0.02):
        return torch.randn(shape, generator=g, device="cuda", dtype=dt) * std

    q_size, kv_size = heads * HEAD_DIM, KV_HEADS * HEAD_DIM
    weights = {"model.embed_tokens.weight": r(VOCAB, hidden),
               "model.norm.weight": 1 + r(hidden)}
    kv = []
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        weights.update({
            p + "self_attn.q_proj.weight": r(q_size, hidden),
            p + "self_attn.k_proj.weight": r(kv_size, hidden),
            p + "self_attn.v_proj.weight": r(kv_size, hidden),
            p + "self_attn.o_proj.weight": r(hidden, q_size),
            p + "self_attn.q_norm.weight": 1 + r(HEAD_DIM),
            p + "self_attn.k_norm.weight": 1 + r(HEAD_DIM),
            p + "mlp.gate_proj.weight": r(ffn, hidden), p + "mlp.up_proj.weight": r(ffn, hidden),
            p + "mlp.down_proj.weight": r(hidden, ffn),
            p + "input_layernorm.weight": 1 + r(hidden),
            p + "post_attention_layernorm.weight": 1 + r(hidden)})
        kv.append((r(pool * PAGE, KV_HEADS, HEAD_DIM, std=1.0),
                   r(pool * PAGE, KV_HEADS, HEAD_DIM, std=1.0)))
    ids = torch.randint(0, VOCAB, (case["rows"],), generator=_gen(seed + 5, "cpu")).tolist()
    return after, pool, tables, weights, kv, ids


# ------------------------------------------------------------------ prepare --

def _cache(pool, kv_heads, dim, key, value, layout, ks=1.0, vs=1.0):
    from tinyvllm.paged_kv import PagedKVCache

    cache = PagedKVCache(num_layers=1, num_blocks=pool, block_size=PAGE, num_kv_heads=kv_heads,
                         head_dim=dim, device="cuda", dtype=key.dtype, k_scale=ks, v_scale=vs,
                         layout=layout)
    cache.key[0].copy_(key)
    cache.value[0].copy_(value)
    return cache


def _csr(tables):
    offsets = [0]
    for t in tables:
        offsets.append(offsets[-1] + len(t))
    return torch.cat(tables).cuda(), torch.tensor(offsets).cuda()


def _metadata(queries, contexts, tables):
    """The runner's eager lowering: decode rows, or prefill items."""
    from tinyvllm.runtime.contracts import MultiQueryMetadata, SingleQueryMetadata

    blocks, offsets = _csr(tables)
    lengths = torch.tensor(contexts).cuda()
    if max(queries) == 1:
        return SingleQueryMetadata(torch.arange(len(queries)).cuda(), blocks, offsets, lengths,
                                   max(contexts)), None
    starts = torch.tensor([0] + queries).cumsum(0).cuda()
    return None, MultiQueryMetadata(starts, blocks, offsets, lengths, max(queries))


def prepare(case, seed):
    return {"decode": _prepare_attention, "prefill": _prepare_attention,
            "pointwise": _prepare_pointwise, "sample": _prepare_sample, "layer": _prepare_layer,
            "step": _prepare_step}[case["kind"]](case, seed)


def _prepare_attention(case, seed):
    queries, contexts, pool, tables, q, k, v, ks, vs = _attention_inputs(case, seed)
    decode, prefill = _metadata(queries, contexts, tables)
    return dict(kind=case["kind"], q=q, out=torch.empty_like(q), scale=case["dim"] ** -0.5,
                cache=_cache(pool, case["kv_heads"], case["dim"], k, v, case["layout"], ks, vs),
                metadata=decode if decode is not None else prefill)


def _prepare_pointwise(case, seed):
    from tinyvllm.layers import RMSNorm, RotaryEmbedding
    from tinyvllm.paged_kv import PagedKVCache

    x = _pointwise_inputs(case, seed)
    dt, n, heads = DTYPES[case["dtype"]], case["tokens"], x["heads"]
    cache = PagedKVCache(num_layers=1, num_blocks=x["pool"], block_size=PAGE,
                         num_kv_heads=KV_HEADS, head_dim=HEAD_DIM, device="cuda", dtype=dt)
    cache.key.zero_()
    cache.value.zero_()
    norm = RMSNorm(x["x"].shape[1], eps=EPS, device="cuda", dtype=dt)
    norm.weight.data.copy_(x["weight"])
    rope = RotaryEmbedding(HEAD_DIM, 2048, base=THETA, device="cuda")(x["positions"], dt)
    q, kv = heads * HEAD_DIM, KV_HEADS * HEAD_DIM
    return dict(kind="pointwise", norm=norm, rope=rope, cache=cache,
                q=x["qkv"][:, :q].view(n, heads, HEAD_DIM),
                k=x["qkv"][:, q:q + kv].view(n, KV_HEADS, HEAD_DIM),
                v=x["qkv"][:, q + kv:].view(n, KV_HEADS, HEAD_DIM), **x_only(x))


def x_only(x):
    return {k: x[k] for k in ("x", "residual", "q_weight", "k_weight", "gate_up", "slots")}


def _prepare_sample(case, seed):
    rows, vocab = case["rows"], case["vocab"]
    g, c = _gen(seed), _gen(seed, "cpu")
    logits = torch.randn((rows, vocab), generator=g, device="cuda") * 2
    # A few likely tokens above the crowd, as a trained head gives.
    likely = torch.randint(0, vocab, (rows, 12), generator=g, device="cuda")
    logits.scatter_(1, likely, 8 + 3 * torch.rand((rows, 12), generator=g, device="cuda"))
    if case["dtype"] != "fp32":
        logits = logits.to(DTYPES[case["dtype"]])

    def pick(values):
        return torch.tensor(values)[torch.randint(0, len(values), (rows,), generator=c)]

    temperature = pick([0.0, 0.6, 0.7, 1.0])
    return dict(kind="sample", logits=logits, temperature=temperature.float().cuda(),
                top_k=pick([0, 20, 50]).long().cuda(),
                top_p=pick([1.0, 0.95, 0.8]).float().cuda(),
                seeds=torch.randint(0, 1 << 40, (rows,), generator=c).cuda(),
                counters=torch.randint(0, 500, (rows,), generator=c).cuda())


def _config(width, layers):
    from tinyvllm.models.qwen3 import Qwen3Config

    hidden, ffn, heads = WIDTHS[width]
    return Qwen3Config(vocab_size=VOCAB, hidden_size=hidden, intermediate_size=ffn,
                       num_hidden_layers=layers, max_position_embeddings=32768,
                       num_attention_heads=heads, num_key_value_heads=KV_HEADS,
                       head_dim=HEAD_DIM, rms_norm_eps=EPS, rope_theta=THETA,
                       tie_word_embeddings=True)


def _prepare_layer(case, seed):
    from tinyvllm.layers import RMSNorm, RotaryEmbedding
    from tinyvllm.models.qwen3 import Qwen3DecoderLayer
    from tinyvllm.runtime.contracts import ModelInput, PagedKVMetadata

    queries, after, pool, tables, positions, slots, w, x = _layer_inputs(case, seed)
    layer = Qwen3DecoderLayer(_config(case["width"], 1), device="meta", dtype=torch.bfloat16)
    layer = layer.to_empty(device="cuda").eval()
    norm = RMSNorm(x["hidden"].shape[1], eps=EPS, device="cuda", dtype=torch.bfloat16)
    for param, name in ((layer.self_attn.qkv_proj.weight, "qkv"), (layer.self_attn.o_proj.weight, "o"),
                        (layer.self_attn.q_norm.weight, "q_norm"),
                        (layer.self_attn.k_norm.weight, "k_norm"),
                        (layer.mlp.gate_up_proj.weight, "gate_up"),
                        (layer.mlp.down_proj.weight, "down"), (layer.input_layernorm.weight, "norm1"),
                        (layer.post_attention_layernorm.weight, "norm2"), (norm.weight, "norm3")):
        param.data.copy_(w[name])
    decode, prefill = _metadata(queries, after, tables)
    positions = positions.cuda()
    rope = RotaryEmbedding(HEAD_DIM, max(after), base=THETA, device="cuda")(positions,
                                                                            torch.bfloat16)
    inputs = ModelInput(input_ids=torch.zeros_like(positions), positions=positions,
                        sample_token_indices=None,
                        kv=PagedKVMetadata(slots.cuda(), decode=decode, prefill=prefill))
    return dict(kind="layer", layer=layer, norm=norm, rope=rope, inputs=inputs,
                hidden=x["hidden"], residual=x["residual"],
                cache=_cache(pool, KV_HEADS, HEAD_DIM, x["key"], x["value"], case["layout"]))


def _prepare_step(case, seed):
    import numpy as np

    from tinyvllm.batch import PreparedBatch, StepMode
    from tinyvllm.models.qwen3 import Qwen3ForCausalLM
    from tinyvllm.request import SamplingParams
    from tinyvllm.runtime.runner import ModelRunner

    after, pool, tables, weights, kv, ids = _step_inputs(case, seed)
    cfg = _config(case["width"], case["layers"])
    model = Qwen3ForCausalLM.random_init(cfg, device="cuda", seed=seed)
    for name, tensor in weights.items():
        model.load_weight(name, tensor)
    rows = case["rows"]
    runner = ModelRunner(model, block_size=PAGE, num_blocks=pool, max_model_len=4096,
                         max_num_seqs=rows, graph_sizes=(rows,), prefill_graph_tokens=0)
    for i, (k, v) in enumerate(kv):
        runner.kv_cache.key[i].copy_(k)
        runner.kv_cache.value[i].copy_(v)
    offsets = [0]
    for t in tables:
        offsets.append(offsets[-1] + len(t))
    slots = [int(t[(n - 1) // PAGE]) * PAGE + (n - 1) % PAGE for t, n in zip(tables, after)]
    requests = tuple(range(rows))
    batch = PreparedBatch(
        plan_id=0, mode=StepMode.DECODE_ONLY, input_ids=tuple(ids),
        positions=tuple(n - 1 for n in after), q_offsets=tuple(range(rows + 1)),
        context_lens_before=tuple(n - 1 for n in after), query_lens=(1,) * rows,
        context_lens_after=tuple(after), sample_token_indices=requests,
        sample_request_ids=requests, sampling_params=(SamplingParams(),) * rows,
        kv_block_size=PAGE, kv_num_blocks=pool,
        kv_block_table_ids=np.asarray(torch.cat(tables)), kv_block_table_offsets=tuple(offsets),
        kv_slot_mapping=np.asarray(slots), request_ids=requests, request_slots=requests,
        kv_table_epochs=requests)
    return dict(kind="step", runner=runner, batch=batch, counters=[0] * rows)


# ---------------------------------------------------------------------- run --

@torch.inference_mode()
def run(state):
    return {"decode": _run_decode, "prefill": _run_prefill, "pointwise": _run_pointwise,
            "sample": _run_sample, "layer": _run_layer, "step": _run_step}[state["kind"]](state)


def _run_decode(s):
    from tinyvllm.kernels.paged_decode import paged_decode_attention

    paged_decode_attention(s["q"], s["cache"], 0, s["metadata"], s["out"], scale=s["scale"])
    return s["out"]


def _run_prefill(s):
    from tinyvllm.kernels.paged_prefill import paged_prefill_attention

    paged_prefill_attention(s["q"], s["cache"], 0, s["metadata"], s["out"], scale=s["scale"])
    return s["out"]


def _run_pointwise(s):
    from tinyvllm.kernels.pointwise import qk_norm_rope_store, silu_and_mul

    normed, merged = s["norm"].add(s["x"], s["residual"])
    cache = s["cache"]
    q, _ = qk_norm_rope_store(s["q"], s["k"], s["v"], s["q_weight"], s["k_weight"], *s["rope"],
                              EPS, EPS, cache.key[0], cache.value[0], s["slots"])
    return dict(normed=normed, merged=merged, q=q, key=cache.key, value=cache.value,
                gated=silu_and_mul(s["gate_up"]))


def _run_sample(s):
    from tinyvllm.kernels.sampling import sample

    return sample(s["logits"], s["temperature"], s["top_k"], s["top_p"], s["seeds"],
                  s["counters"])


def _run_layer(s):
    from tinyvllm.runtime.attention import HipAttention

    attention = HipAttention(s["inputs"], s["cache"])
    out, residual = s["layer"](s["hidden"], s["rope"], residual=s["residual"], layer_idx=0,
                               attention=attention)
    normed, merged = s["norm"].add(out, residual)
    return dict(normed=normed, merged=merged, key=s["cache"].key, value=s["cache"].value)


def _run_step(s):
    # The step samples too; its greedy ids are the logits' argmax, which a
    # rounding decides between near ties of random weights, so the logits stand
    # for them.
    logits, _ = s["runner"].run_and_sample(s["batch"], s["counters"])
    cache = s["runner"].kv_cache
    return dict(logits=logits, key=cache.key, value=cache.value)


# --------------------------------------------------------------------- work --

def _attention_work(queries, contexts, heads, kv_heads, dim, element):
    """K and V of each context once, q and out once; four flops per causal
    (query, key) pair, head and dim."""
    keys = sum(contexts)
    pairs = sum(q * (c - q) + q * (q + 1) / 2 for q, c in zip(queries, contexts))
    return dict(bytes=2 * keys * kv_heads * dim * element + 4 * sum(queries) * heads * dim,
                flops=4 * pairs * heads * dim)


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        if kind == "decode":
            queries, contexts = [1] * case["rows"], [(case["low"] + case["high"]) / 2] * case["rows"]
        else:
            mean = (9 * case["query"] / 16) if case["ragged"] else case["query"]
            queries = [mean] * case["items"]
            contexts = [x + case["history"] for x in queries]
        return _attention_work(queries, contexts, case["heads"], case["kv_heads"], case["dim"],
                               1 if case["cache"] == "fp8" else 2)
    if kind == "pointwise":
        hidden, ffn, heads = WIDTHS[case["width"]]
        per_token = 4 * hidden + 2 * (heads + 2 * KV_HEADS) * HEAD_DIM + HEAD_DIM + 3 * ffn
        return dict(bytes=2 * case["tokens"] * per_token, flops=20 * case["tokens"] * per_token)
    if kind == "sample":
        size = 4 if case["dtype"] == "fp32" else 2
        return dict(bytes=case["rows"] * case["vocab"] * size, flops=4 * case["rows"] * case["vocab"])
    hidden, ffn, heads = WIDTHS[case["width"]]
    weights = (hidden * (heads + 2 * KV_HEADS) * HEAD_DIM + hidden * heads * HEAD_DIM
               + 3 * hidden * ffn)
    query = case.get("query", 1)
    tokens = case["rows"] * query
    mean = (case["low"] + case["high"]) / 2
    attn = _attention_work([query] * case["rows"], [mean] * case["rows"], heads, KV_HEADS,
                           HEAD_DIM, 2)
    if kind == "layer":
        return dict(bytes=2 * weights + attn["bytes"] + 8 * tokens * hidden,
                    flops=2 * weights * tokens + attn["flops"])
    head = VOCAB * hidden
    return dict(bytes=case["layers"] * (2 * weights + attn["bytes"]) + 2 * head
                + 2 * tokens * VOCAB,
                flops=case["layers"] * (2 * weights * tokens + attn["flops"]) + 2 * head * tokens)


def tolerance(case):
    """About four times the distance between two correct evaluations: results
    rounded once to 8 (bf16) or 11 (fp16) bits; a layer and a step round after
    every op, so differences of single roundings add up along the chain."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind in ("decode", "prefill"):
        return {"rel": 8e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}
    if kind == "pointwise":
        return {"rel": 4e-3} if case["dtype"] == "bf16" else {"rel": 5e-4}
    if kind == "layer":
        return {"rel": 1.5e-2}
    return {"rel": 3e-2}


# -------------------------------------------------------------------- exact --

def _attend64(q, key, value, tables, queries, contexts, scale):
    """Causal attention in 64 bits: q [tokens, heads, dim], K/V [slots, kv, dim]."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    group, at = q.shape[1] // key.shape[1], 0
    for table, n, c in zip(tables, queries, contexts):
        slots = _slots(table, c).to(q.device)
        k, v = key[slots].double(), value[slots].double()
        mask = None
        if n > 1:
            allowed = torch.arange(c - n, c, device=q.device)[:, None]
            mask = torch.arange(c, device=q.device)[None, :] > allowed
        for h in range(key.shape[1]):
            x = q[at:at + n, h * group:(h + 1) * group].double().transpose(0, 1)
            s = (x.reshape(-1, x.shape[-1]) @ k[:, h].T).view(group, n, c) * scale
            if mask is not None:
                s.masked_fill_(mask, -math.inf)
            o = torch.softmax(s, -1).reshape(group * n, c) @ v[:, h]
            out[at:at + n, h * group:(h + 1) * group] = o.view(group, n, -1).transpose(0, 1)
        at += n
    return out


def _rms64(x, weight):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _rope64(x, positions):
    half = x.shape[-1] // 2
    freq = THETA ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    angle = positions.double()[:, None, None] * freq
    cos, sin = angle.cos(), angle.sin()
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _layer64(x, residual, w, heads, key, value, slots, positions, tables, queries, after):
    """One decoder layer in 64 bits; returns (MLP output, residual) and writes K, V."""
    tokens, q_size, kv_size = x.shape[0], heads * HEAD_DIM, KV_HEADS * HEAD_DIM
    residual = x if residual is None else x + residual
    qkv = _rms64(residual, w["norm1"]) @ w["qkv"].double().T
    q = _rope64(_rms64(qkv[:, :q_size].view(tokens, heads, HEAD_DIM), w["q_norm"]), positions)
    k = _rope64(_rms64(qkv[:, q_size:q_size + kv_size].view(tokens, KV_HEADS, HEAD_DIM),
                       w["k_norm"]), positions)
    key[slots] = k
    value[slots] = qkv[:, q_size + kv_size:].reshape(tokens, KV_HEADS, HEAD_DIM)
    o = _attend64(q, key, value, tables, queries, after, HEAD_DIM ** -0.5)
    residual = residual + o.reshape(tokens, q_size) @ w["o"].double().T
    gate, up = (_rms64(residual, w["norm2"]) @ w["gate_up"].double().T).chunk(2, -1)
    return (torch.nn.functional.silu(gate) * up) @ w["down"].double().T, residual


@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        queries, contexts, _, tables, q, k, v, ks, vs = _attention_inputs(case, seed)
        return _attend64(q, k.float() if case["cache"] == "fp8" else k,
                         v.float() if case["cache"] == "fp8" else v, tables, queries, contexts,
                         case["dim"] ** -0.5 * ks) * vs
    if kind == "pointwise":
        x = _pointwise_inputs(case, seed)
        n, heads = case["tokens"], x["heads"]
        q_size, kv_size = heads * HEAD_DIM, KV_HEADS * HEAD_DIM
        merged = x["x"].double() + x["residual"].double()
        q = _rms64(x["qkv"][:, :q_size].view(n, heads, HEAD_DIM), x["q_weight"])
        k = _rms64(x["qkv"][:, q_size:q_size + kv_size].view(n, KV_HEADS, HEAD_DIM), x["k_weight"])
        key = torch.zeros((1, x["pool"] * PAGE, KV_HEADS, HEAD_DIM), dtype=torch.float64,
                          device="cuda")
        value = torch.zeros_like(key)
        key[0, x["slots"]] = _rope64(k, x["positions"])
        value[0, x["slots"]] = x["qkv"][:, q_size + kv_size:].double().reshape(n, KV_HEADS, HEAD_DIM)
        gate, up = x["gate_up"].double().chunk(2, -1)
        return dict(normed=_rms64(merged, x["weight"]), merged=merged, q=_rope64(q, x["positions"]),
                    key=key, value=value, gated=torch.nn.functional.silu(gate) * up)
    if kind == "layer":
        queries, after, _, tables, positions, slots, w, x = _layer_inputs(case, seed)
        key, value = x["key"].double(), x["value"].double()
        out, residual = _layer64(x["hidden"].double(), x["residual"].double(), w,
                                 WIDTHS[case["width"]][2], key, value, slots.cuda(),
                                 positions.cuda(), tables, queries, after)
        merged = out + residual
        return dict(normed=_rms64(merged, w["norm3"]), merged=merged, key=key[None],
                    value=value[None])
    if kind == "step":
        after, _, tables, weights, kv, ids = _step_inputs(case, seed)
        embed = weights["model.embed_tokens.weight"]
        x, residual = embed[torch.tensor(ids).cuda()].double(), None
        positions = torch.tensor(after).cuda() - 1
        slots = torch.cat([_slots(t, n, n - 1) for t, n in zip(tables, after)]).cuda()
        keys, values = [], []
        for i, (k, v) in enumerate(kv):
            p = f"model.layers.{i}."
            w = dict(norm1=weights[p + "input_layernorm.weight"],
                     norm2=weights[p + "post_attention_layernorm.weight"],
                     qkv=torch.cat([weights[p + f"self_attn.{n}_proj.weight"] for n in "qkv"]),
                     q_norm=weights[p + "self_attn.q_norm.weight"],
                     k_norm=weights[p + "self_attn.k_norm.weight"],
                     o=weights[p + "self_attn.o_proj.weight"],
                     gate_up=torch.cat([weights[p + f"mlp.{n}_proj.weight"] for n in ("gate", "up")]),
                     down=weights[p + "mlp.down_proj.weight"])
            keys.append(k.double())
            values.append(v.double())
            x, residual = _layer64(x, residual, w, WIDTHS[case["width"]][2], keys[-1], values[-1],
                                   slots, positions, tables, [1] * case["rows"], after)
        logits = _rms64(x + residual, weights["model.norm.weight"]) @ embed.double().T
        return dict(logits=logits, key=torch.stack(keys), value=torch.stack(values))
    return None
