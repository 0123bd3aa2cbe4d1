"""The work by which the speed of this framework is judged: decode steps and prompt
(prefill) calls of one attention layer, a stack of layers, and the Llama-shaped model
around them, each through its public entry point and over the sizes, types and options
that its configurations, tests and benchmark use.

Every case is a dict of plain values; ``kind`` says which entry point it calls:

  "decode"         DRAMAttention(...)(xq, xk, xv, start_pos=, stage="generate"), one token a
                   call, launched from Python as the evaluation harness launches it
  "stack"          AttentionStack.generate, one model step in one HIP graph
  "prefill"        DRAMAttention(...)(xq, xk, xv, start_pos=0, stage="prefill")
  "model_prefill"  Transformer(tokens (1, S), 0)
  "model_decode"   one token: GraphedDecoder.step() (``graph``) as the chat example
                   decodes, or Transformer(token, position) as the evaluation harness does
"""

import math

import torch

from dram_attention_amd import AttentionStack, DRAMAttention, LRUCache
from dram_attention_amd.llama import GraphedDecoder, ModelArgs, Transformer, ffn_hidden_dim

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ESIZE = {"bf16": 2, "fp16": 2, "fp32": 4}

# Decode inputs of one state: a drifting query walked forth and back, so that the drift
# from one call to the next is the same everywhere.  It is longer than the page cache's
# memory (a 128K layer replaces its slots in about 16 steps).
STEPS = 40


def attn(kind, dtype, heads, kv_heads, head_dim, tokens, local, lru, top_k, page=16, **more):
    """``tokens``: of the prompt; the other sizes are DRAMAttention's, in tokens."""
    return dict(kind=kind, dtype=dtype, heads=heads, kv_heads=kv_heads, head_dim=head_dim, tokens=tokens,
                local=local, lru=lru, top_k=top_k, page=page, **more)


def model(kind, dtype, dim, layers, heads, kv_heads, vocab, tokens, local, lru, top_k, page=16, **more):
    return dict(kind=kind, dtype=dtype, dim=dim, layers=layers, heads=heads, kv_heads=kv_heads, vocab=vocab,
                tokens=tokens, local=local, lru=lru, top_k=top_k, page=page, **more)


def listed():
    return [
        # The smallest decode step: an fp32 layer over an 8K prefix, all launch latency.
        dict(attn("decode", "fp32", 8, 2, 64, 9200, 1024, 2048, 512), name="decode fp32 8k"),
        # The prefix fits the page cache: plain attention over a static cache, no selection.
        dict(attn("decode", "bf16", 32, 8, 128, 36848, 4096, 32768, 4096), name="decode bf16 32k static"),
        # The headline decode step: 128K tokens in host memory, a quarter of them cached.
        dict(attn("decode", "bf16", 32, 8, 128, 135152, 4096, 32768, 4096), name="decode bf16 128k"),
        # A ragged mid-size layer in the other 16-bit type: seven query heads to a kv head.
        dict(attn("decode", "fp16", 28, 4, 128, 50021, 1000, 16384, 2048), name="decode fp16 50k ragged"),
        # The largest decode step: 64 query heads over a million tokens.
        dict(attn("decode", "bf16", 64, 8, 128, 1056752, 8192, 65536, 8192), name="decode bf16 1m"),
        # Several layers a step, page streams overlapping the next layers' selection.
        dict(attn("stack", "bf16", 32, 8, 128, 69616, 4096, 16384, 2048, layers=4), name="stack 4 x 64k"),
        # A short prompt: attention over it, and the static cache built from it.
        dict(attn("prefill", "bf16", 32, 8, 128, 4613, 4096, 32768, 4096), name="prefill bf16 4.6k"),
        # The fp32 layer's prompt: attention, page summaries, page store.
        dict(attn("prefill", "fp32", 8, 2, 64, 9200, 1024, 2048, 512), name="prefill fp32 9k"),
        # The headline prompt.
        dict(attn("prefill", "bf16", 32, 8, 128, 135152, 4096, 32768, 4096), name="prefill bf16 132k"),
        # A prompt through the model: projections, rotary embedding, norms, feed-forward.
        dict(model("model_prefill", "bf16", 4096, 2, 32, 8, 128256, 8192, 5120, 2048, 512), name="model prefill 8k"),
        # Chat: one token through the model in one graph, large layers over paged prefixes.
        dict(model("model_decode", "bf16", 4096, 4, 32, 8, 128256, 36848, 4096, 8192, 2048, graph=True),
             name="model decode graph 32k"),
        # Evaluation: one token launched from Python, a small model over an 8K prompt.
        dict(model("model_decode", "bf16", 2048, 4, 16, 4, 32000, 8192, 1088, 2048, 512, graph=False),
             name="model decode eager 8k"),
    ]


def log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "stack", "prefill", "prefill", "model_prefill", "model_decode"])
    page = rng.choice([16, 16, 16, 32])
    heads, kv_heads, head_dim = rng.choice([(8, 2, 64), (16, 4, 64), (32, 8, 128), (24, 8, 128), (28, 4, 128),
                                            (64, 8, 128), (40, 10, 128), (16, 16, 64)])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])

    def caches(prefix):
        """(lru, top_k): an eighth to all of the prefix cached, and up to half of that
        selected, shared out over the query heads of a kv head."""
        lru = max(4 * page, log_uniform(rng, max(prefix // 8, 256), max(prefix, 512)) // page * page)
        return lru, max(page, min(lru // 2 // max(1, heads // kv_heads), 8192) // page * page)

    if kind == "decode":
        local = rng.choice([256, 1000, 1024, 4096])
        prefix = log_uniform(rng, 4096, 400000 if dtype != "fp32" else 60000)
        lru, top_k = caches(prefix)
        return attn(kind, dtype, heads, kv_heads, head_dim, prefix + local, local, lru, top_k, page)
    if kind == "stack":
        local, prefix = rng.choice([512, 1024, 4096]), log_uniform(rng, 8192, 70000)
        lru, top_k = caches(prefix)
        return attn(kind, rng.choice(["bf16", "fp16"]), heads, kv_heads, head_dim, prefix + local, local,
                    min(lru, prefix // 2 // page * page), top_k, page, layers=rng.randint(2, 5))
    if kind == "prefill":
        local = rng.choice([256, 1000, 1024])
        prefix = log_uniform(rng, 1500, 60000 if dtype != "fp32" else 8000)
        lru, top_k = caches(prefix)
        return attn(kind, dtype, heads, kv_heads, head_dim, prefix + local, local, lru, top_k, page)
    head_dim, kv_heads = 128, rng.choice([2, 4, 8])
    heads = kv_heads * rng.choice([1, 2, 4])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    prefix = log_uniform(rng, 1500, 10000 if kind == "model_prefill" else 40000)
    lru, top_k = caches(prefix)
    more = {} if kind == "model_prefill" else {"graph": rng.random() < 0.5}
    return model(kind, dtype, heads * head_dim, rng.randint(1, 3), heads, kv_heads, rng.choice([32000, 50257, 128256]),
                 prefix + 1024, 1024, lru, top_k, page, **more)


# ---- inputs --------------------------------------------------------------------------

def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def prompt_kv(case, g):
    """Keys with outlier channels, values N(0, 1): the workloads' distributions."""
    shape = (case["tokens"], case["kv_heads"], case["head_dim"])
    dtype = DTYPES[case["dtype"]]
    scale = torch.exp(0.5 * torch.randn(shape[1:], generator=g, device="cuda"))
    k = torch.randn(shape, generator=g, device="cuda", dtype=dtype).mul_(scale.to(dtype))
    return k[None], torch.randn(shape, generator=g, device="cuda", dtype=dtype)[None]


def walk(n):
    """Indexes 0 .. n-1 .. 1, for ever."""
    return list(range(n)) + list(range(n - 2, 0, -1))


def drifting_inputs(case, g):
    """STEPS tokens: q_t = 0.9 q_{t-1} + 0.44 N(0, 1), fresh keys and values."""
    dtype, D = DTYPES[case["dtype"]], case["head_dim"]
    q = torch.randn(case["heads"], D, generator=g, device="cuda")
    tokens = []
    for _ in range(STEPS):
        k, v = (torch.randn(1, 1, case["kv_heads"], D, generator=g, device="cuda").to(dtype) for _ in range(2))
        tokens.append((q.to(dtype)[None, None], k, v))
        q = 0.9 * q + 0.44 * torch.randn(q.shape, generator=g, device="cuda")
    return tokens


def layer(case):
    return DRAMAttention(max_output_length=STEPS, lru_hbm_cache_size=case["lru"], local_cache_size=case["local"],
                         page_size=case["page"], top_k=case["top_k"], n_kv_heads=case["kv_heads"],
                         head_dim=case["head_dim"], device="cuda", dtype=DTYPES[case["dtype"]])


def transformer(case, seed):
    torch.manual_seed(seed)
    args = ModelArgs(dim=case["dim"], n_layers=case["layers"], n_heads=case["heads"], n_kv_heads=case["kv_heads"],
                     vocab_size=case["vocab"], multiple_of=1024, ffn_dim_multiplier=1.3, use_scaled_rope=True,
                     lru_hbm_cache_size=case["lru"], local_cache_size=case["local"], cache_page_size=case["page"],
                     cache_top_k=case["top_k"], max_output_length=STEPS, max_seq_len=case["tokens"] + STEPS,
                     dtype=DTYPES[case["dtype"]])
    return Transformer(args, device="cuda")


def prepare(case, seed):
    kind, g = case["kind"], generator(seed)
    state = {"case": case, "pass": 0}
    if kind == "decode":
        state["layer"] = layer(case)
        state["layer"].init_cache(*prompt_kv(case, g))
        state["tokens"] = drifting_inputs(case, g)
    elif kind == "stack":
        layers = [layer(case) for _ in range(case["layers"])]
        for m in layers:
            m.init_cache(*prompt_kv(case, g))
        rows = [drifting_inputs(case, g) for _ in layers]
        # one row per step and layer, [query | key | value], fetched by one copy a step
        state["rows"] = torch.stack([torch.stack([torch.cat([x.flatten() for x in r[t]]) for r in rows])
                                     for t in range(STEPS)])
        state["positions"] = (torch.arange(STEPS, device="cuda") + case["tokens"]).to(torch.int32)[:, None]
        state["row"], state["position"] = state["rows"][0].clone(), state["positions"][0].clone()
        stack = AttentionStack(layers)
        Hq, Hkv, D = case["heads"], case["kv_heads"], case["head_dim"]
        q, k, v = (x.unsqueeze(0).unsqueeze(0) for x in state["row"].split([Hq * D, Hkv * D, Hkv * D], dim=1))

        def step():
            return stack.generate([q[:, :, i].view(1, 1, Hq, D) for i in range(len(layers))],
                                  [k[:, :, i].view(1, 1, Hkv, D) for i in range(len(layers))],
                                  [v[:, :, i].view(1, 1, Hkv, D) for i in range(len(layers))], state["position"])

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()                          # sizes the workspaces
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["stack"], state["graph"] = stack, torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = step()
    elif kind == "prefill":
        state["layer"] = layer(case)
        state["k"], state["v"] = prompt_kv(case, g)
        state["q"] = torch.randn(1, case["tokens"], case["heads"], case["head_dim"], generator=g, device="cuda",
                                 dtype=DTYPES[case["dtype"]])
    elif kind == "model_prefill":
        state["model"] = transformer(case, seed)
        state["prompt"] = torch.randint(0, case["vocab"], (1, case["tokens"]), generator=g, device="cuda")
    else:
        state["model"] = m = transformer(case, seed)
        for block in m.layers:
            block.attention.dram_attention.init_cache(
                *prompt_kv(dict(case, head_dim=case["dim"] // case["heads"]), g))
        # A text's successive queries resemble each other; random weights would make them
        # unrelated and every page a miss.  The tokens fed here have embeddings that
        # drift as the layers' queries do in the other cases.
        x = torch.randn(case["dim"], generator=g, device="cuda")
        for t in range(STEPS):
            with torch.no_grad():
                m.tok_embeddings.weight[t] = x
            x = 0.9 * x + 0.44 * torch.randn(x.shape, generator=g, device="cuda")
        state["tokens"] = torch.arange(STEPS, device="cuda").view(STEPS, 1, 1)
        if case["graph"]:
            state["positions"] = (torch.arange(STEPS, device="cuda") + case["tokens"]).to(torch.int32)[:, None]
            state["decoder"] = GraphedDecoder(m, case["tokens"], first_token=1)
            state["decoder"].step()         # eager: sizes the workspaces
            state["decoder"].step()         # captures
    return state


# ---- one pass ------------------------------------------------------------------------

def cache_state(m, prompt=False):
    """What a call leaves behind in a layer: appended rows, page maps, access times and
    the pages in their slots; after a prompt also the page summaries and the page store."""
    state = {"cache_k": m.cache_k, "cache_v": m.cache_v}
    lru = m.lru_cache
    if isinstance(lru, LRUCache):
        state.update(slots=lru.hbm_kv_cache, slot_of_page=lru.dram_page_to_hbm_page_mapping,
                     page_of_slot=lru.hbm_page_to_dram_page_mapping, access_time=lru.page_access_time)
        if prompt:
            state.update(summaries=lru.top_k_selector.chunk_min_max, store=lru.dram_kv_cache)
    elif prompt:
        state.update(prefix_k=lru.k_cache, prefix_v=lru.v_cache)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    order = walk(STEPS)
    t = order[state["pass"] % len(order)]
    state["pass"] += 1
    if kind == "decode":
        xq, xk, xv = state["tokens"][t]
        m = state["layer"]
        out = m(xq, xk, xv, start_pos=case["tokens"] + t, stage="generate")
        return {"out": out, "state": cache_state(m)}
    if kind == "stack":
        state["row"].copy_(state["rows"][t])
        state["position"].copy_(state["positions"][t])
        state["graph"].replay()
        return {"out": state["out"], "state": [cache_state(m) for m in state["stack"].layers]}
    if kind == "prefill":
        m = state["layer"]
        out = m(state["q"], state["k"], state["v"], start_pos=0, stage="prefill")
        return {"out": out, "state": cache_state(m, prompt=True)}
    attentions = [block.attention.dram_attention for block in state["model"].layers]
    if kind == "model_prefill":
        logits = state["model"](state["prompt"], 0)
    elif case["graph"]:
        decoder = state["decoder"]
        decoder.token.copy_(state["tokens"][t])
        decoder.pos.copy_(state["positions"][t])
        logits = decoder.step()
    else:
        logits = state["model"](state["tokens"][t], case["tokens"] + t)
    # (of the page cache only what the prompt or the token wrote: which pages are best is
    # decided by scores that lie within one rounding of each other)
    return {"logits": logits, "state": [{"cache_k": m.cache_k, "cache_v": m.cache_v} for m in attentions]}


# ---- what a pass cannot do without ---------------------------------------------------

def prefix_tokens(case):
    return (case["tokens"] - case["local"] + case["page"]) // case["page"] * case["page"]


def attention_decode_work(case, kv_heads, heads, head_dim):
    """One decode step of one layer: page summaries once, resident and local keys and
    values once.  Pages that miss come on top, as many as the inputs ask for."""
    e, prefix = ESIZE[case["dtype"]], prefix_tokens(case)
    paged = prefix > case["lru"]
    resident = case["lru"] // case["page"] * case["page"] if paged else prefix
    attended = resident + case["tokens"] - prefix + STEPS // 2
    moved = attended * kv_heads * 2 * head_dim * e + 2 * heads * head_dim * e
    flops = 4 * attended * heads * head_dim
    if paged:
        moved += prefix // case["page"] * kv_heads * 2 * head_dim * e
        flops += 4 * prefix // case["page"] * heads * head_dim
    return moved, flops


def attention_prefill_work(case, kv_heads, heads, head_dim):
    """Causal attention over the prompt and the caches built from it."""
    e, S, prefix = ESIZE[case["dtype"]], case["tokens"], prefix_tokens(case)
    row = kv_heads * 2 * head_dim * e
    moved = 2 * S * heads * head_dim * e + S * row + (S - prefix) * row
    if prefix > case["lru"]:
        moved += prefix * row + case["lru"] * row + prefix // case["page"] * row
    return moved, 2 * S * S * heads * head_dim


def work(case):
    kind = case["kind"]
    if kind in ("decode", "stack", "prefill"):
        one = attention_prefill_work if kind == "prefill" else attention_decode_work
        moved, flops = one(case, case["kv_heads"], case["heads"], case["head_dim"])
        n = case.get("layers", 1)
        return {"bytes": n * moved, "flops": n * flops}
    e, dim, heads, kv_heads = ESIZE[case["dtype"]], case["dim"], case["heads"], case["kv_heads"]
    D = dim // heads
    weights = dim * D * (2 * heads + 2 * kv_heads) + 3 * dim * ffn_hidden_dim(dim, 1024, 1.3)
    rows = case["tokens"] if kind == "model_prefill" else 1
    one = attention_prefill_work if kind == "model_prefill" else attention_decode_work
    moved, flops = one(case, kv_heads, heads, D)
    # queries, keys, values and attention's output stay between the parts of a layer
    moved = case["layers"] * (moved + weights * e) + case["vocab"] * (dim * e + 4) + rows * (dim * e + 8)
    return {"bytes": moved, "flops": case["layers"] * (flops + 2 * rows * weights) + 2 * dim * case["vocab"]}


def tolerance(case):
    """About four times the distance to the same call in a wider type.  Attention of one
    layer against float64 over the same keys: 2.3e-3 (largest 1.8e-2) in bf16, 2.6e-4
    in fp16, 8.6e-7 (1.5e-5) in fp32, with room for longer sums.  Logits of the model
    against its float32 copy, static caches: 5.3e-3 (2.2e-2) in bf16, 7e-4 (2.7e-3) in
    fp16.  Page maps of a layer stay the same whole numbers."""
    if case["kind"].startswith("model"):
        return {"bf16": {"rel": 0.02, "max": 0.1}, "fp16": {"rel": 3e-3, "max": 0.012}}[case["dtype"]]
    return {"bf16": {"rel": 0.01, "max": 0.08}, "fp16": {"rel": 1.2e-3, "max": 0.01},
            "fp32": {"rel": 1e-5, "max": 1e-4}}[case["dtype"]]
