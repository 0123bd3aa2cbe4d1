"""configs[3] in small: several attention layers of the 128K shape stepped as one model
step, with layer i's page stream overlapping the selection of the layers after it.

Every layer is compared with its own CPU oracle at every step (request list, maps,
access times, hit mask, slot payload bit for bit; output within the bf16 tolerance),
and the pipelined order must give the same bits as stepping the layers one by one.
The pipelined model step is captured into one HIP graph and replayed, with the
position on the device, as a serving loop would run it."""

import pytest
import torch

from dram_attention_amd.synthetic import WORKLOADS, DecodeInputs, make_prompt
from oracle import dram_attention_oracle as O
from tests.parity import check_invariants, check_step
from tests.util import same

pytestmark = pytest.mark.gpu
DEV = "cuda"


def build(w, n_layers, seed0, max_out):
    from dram_attention_amd import DRAMAttention

    layers, oracles, feeds = [], [], []
    for li in range(n_layers):
        prompt = make_prompt(w, seed0 + li)
        m = DRAMAttention(max_out, w.lru_tokens, w.local_cache, w.page_size, w.top_k_tokens,
                          w.n_kv_heads, w.head_dim, device=DEV, dtype=w.dtype)
        m.init_cache(prompt.k.to(DEV), prompt.v.to(DEV))
        o = O.DecodeOracle(max_out, w.lru_tokens, w.local_cache, w.page_size, w.top_k_tokens,
                           w.n_kv_heads, w.head_dim, dtype=w.dtype)
        o.init_cache(prompt.k, prompt.v)
        layers.append(m)
        oracles.append(o)
        feeds.append(DecodeInputs(w, prompt.q0, seed0 + li))
        print(f"stack test: layer {li} built", flush=True)
    return layers, oracles, feeds


@pytest.mark.parametrize("shape", ["scaled", "128k"])
def test_pipelined_stack_matches_oracles_and_serial_order(shape):
    from dram_attention_amd import AttentionStack, DRAMAttention

    if shape == "128k":
        w, n_layers, steps = WORKLOADS["128k"], 4, 3       # configs[3]'s layer, four of them
    else:
        w = WORKLOADS["128k"].scaled(dram_tokens=16384, local_cache=1024, lru_tokens=4096,
                                     top_k_tokens=1024)
        n_layers, steps = 6, 5
    layers, oracles, feeds = build(w, n_layers, 40, steps)
    stack = AttentionStack(layers, pipelined=True)
    # the same layers again, stepped one by one on one stream
    serial = []
    for li in range(n_layers):
        prompt = make_prompt(w, 40 + li)
        m = DRAMAttention(steps, w.lru_tokens, w.local_cache, w.page_size, w.top_k_tokens,
                          w.n_kv_heads, w.head_dim, device=DEV, dtype=w.dtype)
        m.init_cache(prompt.k.to(DEV), prompt.v.to(DEV))
        serial.append(m)
    serial_stack = AttentionStack(serial, pipelined=False)

    host = [[f.next() for f in feeds] for _ in range(steps)]           # [step][layer] -> (q, k, v)
    bufs = [tuple(torch.empty_like(x, device=DEV) for x in host[0][li]) for li in range(n_layers)]
    pos = torch.tensor([w.prompt_tokens], dtype=torch.int32, device=DEV)

    def feed(t):
        for li in range(n_layers):
            for dst, src in zip(bufs[li], host[t][li]):
                dst.copy_(src)

    def model_step():
        return stack.generate([b[0] for b in bufs], [b[1] for b in bufs], [b[2] for b in bufs], pos)

    def check(t, outs):
        want_serial = serial_stack.generate(*[[x[i].to(DEV) for x in host[t]] for i in range(3)],
                                            w.prompt_tokens + t)
        torch.cuda.synchronize()
        for li in range(n_layers):
            q, k, v = host[t][li]
            check_step(layers[li], oracles[li], q, k, v, w.prompt_tokens + t, outs[li], t, 2e-2, 1e-2)
            assert same(outs[li], want_serial[li]), f"layer {li} step {t}: pipelined vs serial order"
            assert same(layers[li].lru_cache.hbm_kv_cache, serial[li].lru_cache.hbm_kv_cache)
            assert same(layers[li].lru_cache.page_access_time, serial[li].lru_cache.page_access_time)
            assert layers[li].lru_cache.last_miss_counts().sum().item() > 0

    # step 0 eagerly (resolves the pinned mappings, sizes the workspaces)
    feed(0)
    outs = model_step()
    check(0, outs)
    pos += 1
    torch.cuda.synchronize()
    # the rest as one captured model step, replayed
    graph = torch.cuda.CUDAGraph()
    feed(1)
    with torch.cuda.graph(graph):
        outs = model_step()
        pos += 1
    for t in range(1, steps):
        feed(t)
        graph.replay()
        torch.cuda.synchronize()
        assert pos.item() == w.prompt_tokens + t + 1
        check(t, outs)


def test_stack_of_32_full_size_layers_by_properties():
    """configs[3] at its stated depth: 32 layers of the 128K shape (17 GB of pinned pages),
    one model step per HIP graph, 9 decode steps.  No CPU walk: every layer of the
    pipelined stack is held to the size-independent properties of a step (selection
    ordered and maximal, maps mutually inverse, slot payload = mapped page, attention
    against a dense fp32 softmax on the GPU), and to the bits of a second stack over the
    same prompts whose layers are stepped one after the other on one stream."""
    from dram_attention_amd import AttentionStack, DRAMAttention

    w, n_layers, steps = WORKLOADS["128k"], 32, 9
    Hq, Hkv, D = w.n_q_heads, w.n_kv_heads, w.head_dim
    g = torch.Generator(device=DEV).manual_seed(77)
    piped, serial, stores = [], [], []
    for li in range(n_layers):
        # the workload's distributions drawn on the GPU: K ~ N(0,1) x per-channel lognormal(0, 0.5)
        k = torch.randn(w.prompt_tokens, Hkv, D, generator=g, device=DEV)
        k *= torch.exp(0.5 * torch.randn(Hkv, D, generator=g, device=DEV))
        k = k.to(w.dtype)[None]
        v = torch.randn(w.prompt_tokens, Hkv, D, generator=g, device=DEV).to(w.dtype)[None]
        for group in (piped, serial):
            m = DRAMAttention(steps, w.lru_tokens, w.local_cache, w.page_size, w.top_k_tokens,
                              Hkv, D, device=DEV, dtype=w.dtype)
            m.init_cache(k, v)
            group.append(m)
        stores.append(piped[-1].lru_cache.dram_kv_cache.to(DEV))
        del k, v
        if (li + 1) % 8 == 0:
            print(f"stack test: {li + 1} of {n_layers} layer pairs built", flush=True)
    stack, serial_stack = AttentionStack(piped, pipelined=True), AttentionStack(serial, pipelined=False)
    # drifting queries as in the workload: q_t = 0.9 q_{t-1} + 0.44 N(0,1), per layer
    q = torch.randn(n_layers, Hq, D, generator=g, device=DEV)
    feeds = []
    for t in range(steps):
        if t:
            q = 0.9 * q + 0.44 * torch.randn(n_layers, Hq, D, generator=g, device=DEV)
        feeds.append((q.to(w.dtype), torch.randn(n_layers, Hkv, D, generator=g, device=DEV).to(w.dtype),
                      torch.randn(n_layers, Hkv, D, generator=g, device=DEV).to(w.dtype)))
    bufs = tuple(torch.empty_like(x) for x in feeds[0])
    pos = torch.tensor([w.prompt_tokens], dtype=torch.int32, device=DEV)

    def split(x):
        return [x[li][None, None] for li in range(n_layers)]

    def model_step():
        return stack.generate(split(bufs[0]), split(bufs[1]), split(bufs[2]), pos)

    def check(t, outs):
        want = serial_stack.generate(*[split(x) for x in feeds[t]], w.prompt_tokens + t)
        torch.cuda.synchronize()
        missed = 0
        for li in range(n_layers):
            check_invariants(piped[li], w, *[x[li][None, None] for x in feeds[t]], outs[li], t,
                             stores[li])
            assert same(outs[li], want[li]), f"layer {li} step {t}: pipelined vs serial order"
            assert same(piped[li].lru_cache.hbm_kv_cache, serial[li].lru_cache.hbm_kv_cache)
            assert same(piped[li].lru_cache.page_access_time, serial[li].lru_cache.page_access_time)
            missed += piped[li].lru_cache.last_miss_counts().sum().item()
        assert missed > n_layers * 100          # the steps really paged

    for dst, src in zip(bufs, feeds[0]):
        dst.copy_(src)
    outs = model_step()                         # step 0 eagerly: pinned mappings, workspaces
    check(0, outs)
    pos += 1
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = model_step()
        pos += 1
    for t in range(1, steps):
        for dst, src in zip(bufs, feeds[t]):
            dst.copy_(src)
        graph.replay()
        torch.cuda.synchronize()
        assert pos.item() == w.prompt_tokens + t + 1
        check(t, outs)
        print(f"stack test: step {t} of {steps - 1} checked", flush=True)


def test_stack_argument_checks_and_short_stacks():
    from dram_attention_amd import AttentionStack

    w = WORKLOADS["128k"].scaled(dram_tokens=4096, local_cache=256, lru_tokens=1024, top_k_tokens=256)
    layers, oracles, feeds = build(w, 1, 60, 2)
    stack = AttentionStack(layers)
    q, k, v = feeds[0].next()
    with pytest.raises(ValueError):
        stack.generate([q.to(DEV)], [k.to(DEV)], [], w.prompt_tokens)
    (out,) = stack.generate([q.to(DEV)], [k.to(DEV)], [v.to(DEV)], w.prompt_tokens)
    check_step(layers[0], oracles[0], q, k, v, w.prompt_tokens, out, 0, 2e-2, 1e-2)


@pytest.mark.parametrize("n,dtype,heads,sizes", [
    (2, torch.float32, (8, 2, 64), None),
    (8, torch.bfloat16, (8, 2, 64), None), (9, torch.float16, (8, 2, 64), None),   # a batch of launches, one more
    (3, torch.bfloat16, (16, 2, 128), None), (2, torch.float16, (12, 2, 128), None), (2, torch.float32, (4, 4, 128), None),
    # head sizes whose scores, or scores and page streams, go layer by layer
    (3, torch.bfloat16, (8, 2, 32), None), (2, torch.float32, (8, 2, 32), None), (3, torch.float16, (8, 2, 256), None),
    (3, torch.bfloat16, (8, 2, 64), (200, 200, 216)),                              # layers of different sizes
])
def test_layers_stepped_by_one_call_equal_layers_stepped_alone(n, dtype, heads, sizes):
    """Bits of the serial order for every layer, its caches and what its next step starts from."""
    from dram_attention_amd import AttentionStack, DRAMAttention

    Hq, Hkv, D = heads
    S = 1500
    g = torch.Generator(device=DEV).manual_seed(n)

    def rand(*shape):
        return torch.randn(*shape, device=DEV, generator=g).to(dtype)

    stacks = []
    prompts = [(rand(1, S, Hkv, D), rand(1, S, Hkv, D)) for _ in range(n)]
    for pipelined in (True, False):
        layers = [DRAMAttention(6, 800, local, 16, 96, Hkv, D, device=DEV, dtype=dtype)
                  for local in sizes or [200] * n]
        for m, (k, v) in zip(layers, prompts):
            m.init_cache(k, v)
        stacks.append(AttentionStack(layers, pipelined=pipelined))
    together = []
    inner = stacks[0]._together
    stacks[0]._together = lambda *a: together.append(inner(*a)) or together[-1]
    for t in range(4):
        xqs, xks, xvs = ([rand(1, 1, h, D) for _ in range(n)] for h in (Hq, Hkv, Hkv))
        pos = S + t if t % 2 else torch.tensor([S + t], dtype=torch.int32, device=DEV)
        got, want = (s.generate(xqs, xks, xvs, pos) for s in stacks)
        assert (together[t] is None) == (sizes is not None)
        for a, b, x, y in zip(stacks[0].layers, stacks[1].layers, got, want):
            assert same(x, y) and same(a.cache_k, b.cache_k) and same(a.cache_v, b.cache_v)
            for name in ("hbm_kv_cache", "page_access_time", "dram_page_to_hbm_page_mapping",
                         "hbm_page_to_dram_page_mapping", "current_step"):
                assert same(getattr(a.lru_cache, name), getattr(b.lru_cache, name)), (t, name)


def stepped_blocks(n, dtype, heads, S=1500):
    """Two sets of n layers over the same prompts, and for each layer of either set the argument block of a step, as
    a list in the order of the struct, and the output it points at; the partial results start out as NaN."""
    from dram_attention_amd import DRAMAttention, _lib

    Hq, Hkv, D = heads
    g = torch.Generator(device=DEV).manual_seed(n + D)

    def rand(*shape):
        return torch.randn(*shape, device=DEV, generator=g).to(dtype)

    prompts = [(rand(1, S, Hkv, D), rand(1, S, Hkv, D)) for _ in range(n)]
    tokens = [(rand(1, 1, Hq, D), rand(1, 1, Hkv, D), rand(1, 1, Hkv, D)) for _ in range(n)]
    sets = []
    for _ in range(2):
        layers, blocks, outs = [], [], []
        for (k, v), (xq, xk, xv) in zip(prompts, tokens):
            m = DRAMAttention(6, 800, 200, 16, 96, Hkv, D, device=DEV, dtype=dtype)
            m.init_cache(k, v)
            args, out = m._step_args(xq, xk, xv, S)
            m._workspace.fill_(float("nan"))
            layers.append(m)
            blocks.append(list(_lib.DECODE_STEP_ARGS.unpack(args)))
            outs.append(out)
        sets.append((layers, blocks, outs))
    torch.cuda.synchronize()
    return sets, tokens


def step_state(m):
    """What a step leaves behind in a layer."""
    lru = m.lru_cache
    return [m.cache_k, m.cache_v, lru.hbm_kv_cache, lru.page_access_time, lru.dram_page_to_hbm_page_mapping,
            lru.hbm_page_to_dram_page_mapping, lru.current_step]


@pytest.mark.parametrize("dtype,heads", [(torch.float32, (8, 2, 64)), (torch.bfloat16, (16, 2, 128))])
@pytest.mark.parametrize("appends", [(False, True, True), (True, False, True)])
def test_blocks_with_and_without_a_new_token_in_one_call(dtype, heads, appends):
    """The C entry: layers that append a token next to layers that do not, with an empty local window, the edge of a
    chunk; the outputs and caches of a call per block."""
    from dram_attention_amd import _lib

    lib, pack = _lib.load(), _lib.DECODE_STEP_ARGS.pack
    ((layers, blocks, outs), (alone, single, wants)), _tokens = stepped_blocks(3, dtype, heads)
    for block in blocks + single:
        block[28] = 0                                        # cache_len
    for i, append in enumerate(appends):
        if not append:
            blocks[i][1:3] = single[i][1:3] = [0, 0]         # new_k, new_v
    args = b"".join(pack(*b) for b in blocks)
    assert lib.da_decode_steps_supported(args, 3, len(args))
    stream = _lib.stream_ptr(outs[0].device)
    _lib.check(lib.da_decode_steps(args, 3, len(args), stream), "steps")
    for b in single:
        _lib.check(lib.da_decode_step(pack(*b), len(args) // 3, stream), "step")
    for i in range(3):
        assert same(outs[i], wants[i]), i
        assert not outs[i].isnan().any()
        assert all(same(a, b) for a, b in zip(step_state(layers[i]), step_state(alone[i]))), i


@pytest.mark.parametrize("field,value", [(4, 0), (5, 0), (6, 0), (8, 0), (18, 0), (19, 0), (40, 64)],
                         ids=["minmax", "scores", "idx", "access_time", "lru_workspace", "dram", "score_flags"])
def test_a_bad_block_is_refused_before_any_layer_steps(field, value):
    """Nine blocks, one more than a batch of launches, the last one not usable: an error and nothing changed."""
    from dram_attention_amd import _lib

    lib, n = _lib.load(), 9
    ((layers, blocks, outs), _), _tokens = stepped_blocks(n, torch.bfloat16, (8, 2, 64))
    blocks[-1][field] = value
    for out in outs:
        out.fill_(-7.0)
    before = [[t.clone() for t in step_state(m)] for m in layers]
    args = b"".join(_lib.DECODE_STEP_ARGS.pack(*b) for b in blocks)
    rc = lib.da_decode_steps(args, n, len(args), _lib.stream_ptr(outs[0].device))
    torch.cuda.synchronize()
    assert rc == -1 and lib.da_last_error_string()
    for m, state, out in zip(layers, before, outs):
        assert all(same(a, b) for a, b in zip(step_state(m), state)) and (out == -7.0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_blocks_of_other_score_flags_and_query_strides_in_one_call(dtype):
    """The C entry: a layer whose page bounds are not said to be ordered, and one whose query rows lie apart; the
    results of a call per block."""
    from dram_attention_amd import _lib

    lib, pack = _lib.load(), _lib.DECODE_STEP_ARGS.pack
    ((layers, blocks, outs), (alone, single, wants)), tokens = stepped_blocks(3, dtype, (8, 2, 64))
    apart = torch.full((8, 128), float("nan"), dtype=dtype, device=DEV)
    apart[:, :64] = tokens[2][0][0, 0]
    for some in (blocks, single):
        some[1][40] &= 1                                     # DA_SCORE_ROUND alone
        some[2][0], some[2][25] = apart.data_ptr(), 128      # q, q_head_stride
    assert blocks[0][40] != blocks[1][40]
    args = b"".join(pack(*b) for b in blocks)
    assert lib.da_decode_steps_supported(args, 3, len(args))
    stream = _lib.stream_ptr(outs[0].device)
    _lib.check(lib.da_decode_steps(args, 3, len(args), stream), "steps")
    for b in single:
        _lib.check(lib.da_decode_step(pack(*b), len(args) // 3, stream), "step")
    for i in range(3):
        assert same(outs[i], wants[i]), i
        assert all(same(a, b) for a, b in zip(step_state(layers[i]), step_state(alone[i]))), i
