"""The Llama-shaped model around the attention path on the GPU against its CPU
restatement, and graph-captured decoding against eager decoding."""

import pytest
import torch

from dram_attention_amd import llama as L
from oracle import llama_oracle as M

pytestmark = pytest.mark.gpu


def small_args(dtype, **kw):
    base = dict(dim=256, n_layers=3, n_heads=8, n_kv_heads=2, vocab_size=257, multiple_of=32,
                ffn_dim_multiplier=1.3, rope_theta=500000.0, use_scaled_rope=True,
                lru_hbm_cache_size=256, local_cache_size=128, cache_page_size=16,
                cache_top_k=128, max_output_length=16, max_seq_len=1100, dtype=dtype)
    base.update(kw)
    return L.ModelArgs(**base)


def build(args, seed):
    torch.manual_seed(seed)
    model = L.Transformer(args, device="cuda")
    # norms away from their all-ones start, so that a dropped weight shows
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("norm.weight"):
                p.copy_(1.0 + 0.1 * torch.randn_like(p))
    return model


def test_fp32_model_matches_cpu_restatement():
    args = small_args(torch.float32)
    model = build(args, 0)
    oracle = M.LlamaOracle(args, model.state_dict())
    g = torch.Generator().manual_seed(1)
    prompt = torch.randint(0, args.vocab_size, (1, 1000), generator=g)
    got = model(prompt.cuda(), 0).cpu()
    want = oracle.forward(prompt, 0)
    assert got.shape == want.shape == (1, 1, args.vocab_size)
    scale = want.abs().max().item()
    assert torch.allclose(got, want, atol=2e-4 * scale, rtol=1e-3), (got - want).abs().max()
    for layer, o in zip(model.layers, oracle.layers):
        assert o.uses_lru and layer.attention.dram_attention.dram_kv_cache_size == 880
    pos = prompt.shape[1]
    for t in range(args.max_output_length - 1):
        token = want.argmax(-1)                      # both sides are fed the same token
        got = model(token.cuda(), pos).cpu()
        want = oracle.forward(token, pos)
        for i, (layer, o) in enumerate(zip(model.layers, oracle.layers)):
            sel = layer.attention.dram_attention.lru_cache._topk_idx.cpu()
            assert torch.equal(sel, o.last_idx), f"page selection, layer {i}, step {t}"
        assert torch.allclose(got, want, atol=2e-4 * scale, rtol=1e-3), \
            (t, (got - want).abs().max().item())
        assert got.argmax(-1).item() == want.argmax(-1).item()
        pos += 1


def test_device_position_equals_host_position():
    args = small_args(torch.bfloat16)
    a, b = build(args, 2), build(args, 2)
    g = torch.Generator().manual_seed(3)
    prompt = torch.randint(0, args.vocab_size, (1, 700), generator=g).cuda()
    la, lb = a(prompt, 0), b(prompt, 0)
    assert torch.equal(la, lb)
    pos = torch.tensor([700], dtype=torch.int32, device="cuda")
    for t in range(6):
        token = la.argmax(-1)
        la = a(token, 700 + t)
        lb = b(token, pos)
        pos += 1
        assert torch.equal(la, lb), f"step {t}"


def test_graphed_greedy_decoding_equals_eager():
    args = small_args(torch.bfloat16)
    a, b = build(args, 4), build(args, 4)
    g = torch.Generator().manual_seed(5)
    prompt = torch.randint(0, args.vocab_size, (1, 900), generator=g).cuda()
    first = a(prompt, 0).argmax(-1).item()
    assert b(prompt, 0).argmax(-1).item() == first
    dec = L.GraphedDecoder(b, 900, first)
    token = torch.tensor([[first]], device="cuda")
    for t in range(10):
        want = a(token, 900 + t)
        got = dec.step()
        torch.cuda.synchronize()
        assert torch.equal(got, want), f"step {t}"
        token = want.argmax(-1)
        assert torch.equal(dec.token, token)
    assert dec.graph is not None and dec.pos.item() == 910


def test_layer_files_feed_the_model(tmp_path):
    from dram_attention_amd import save_layer_cache

    args = small_args(torch.bfloat16)
    a, b = build(args, 6), build(args, 6)
    g = torch.Generator().manual_seed(7)
    prompt = torch.randint(0, args.vocab_size, (1, 640), generator=g).cuda()
    la = a(prompt, 0)
    # capture every layer's prompt K/V the way the chat example's prefill phase does
    kv = []
    hooks = [layer.attention.dram_attention.register_forward_pre_hook(
        lambda mod, inp, store=kv: store.append((inp[1].cpu(), inp[2].cpu())))
        for layer in b.layers]
    b(prompt, 0)
    for h in hooks:
        h.remove()
    for i, (k, v) in enumerate(kv):
        save_layer_cache(str(tmp_path), i, k, v)
    c = build(args, 6)
    assert c.init_cache_from_files(str(tmp_path)) == 640
    token = la.argmax(-1)
    assert torch.equal(c(token, 640), a(token, 640))


def test_model_variants_full_quest_and_quest_oracle():
    """The reference's comparison models on the same kernels.  "full" keeps the whole
    prefix in HBM behind the static cache (evaluation/full-attention/model.py:201-215):
    its logits follow the CPU restatement of the model with a cache budget that holds
    everything.  "quest" attends over the selected pages only
    (evaluation/quest/model.py:263-316; the attention itself is checked against a dense
    computation in test_gpu_module.py): here, that the model runs it in every layer and
    that it sees fewer tokens than "dram" does.  "quest_oracle" is "quest" with pages
    ranked by their best token (evaluation/quest-top-k-oracle/model.py:267-275; the
    selector is checked in test_gpu_module.py)."""
    from dram_attention_amd import DummyCache, LRUCache
    from dram_attention_amd.topk_selector import TokenMaxTopKSelector

    g = torch.Generator().manual_seed(3)
    prompt = torch.randint(0, 257, (1, 1000), generator=g)
    args = small_args(torch.float32, attention_variant="full")
    model = build(args, 0)
    oracle = M.LlamaOracle(small_args(torch.float32, lru_hbm_cache_size=1100), model.state_dict())
    got, want = model(prompt.cuda(), 0).cpu(), oracle.forward(prompt, 0)
    scale = want.abs().max().item()
    pos = 1000
    for t in range(5):
        assert torch.allclose(got, want, atol=2e-4 * scale, rtol=1e-3), (t, (got - want).abs().max())
        token = want.argmax(-1)
        got, want = model(token.cuda(), pos).cpu(), oracle.forward(token, pos)
        pos += 1
    for layer, o in zip(model.layers, oracle.layers):
        assert isinstance(layer.attention.dram_attention.lru_cache, DummyCache) and not o.uses_lru
    # 8 pages per query head, 32 requests per kv head, 32 slots
    outs = {}
    for variant in ("dram", "quest", "quest_oracle"):
        model = build(small_args(torch.float32, attention_variant=variant, lru_hbm_cache_size=512), 0)
        out = model(prompt.cuda(), 0)
        for layer in model.layers:
            a = layer.attention.dram_attention
            assert isinstance(a.lru_cache, LRUCache)
            assert a.attention_scope == ("resident" if variant == "dram" else "selected")
            assert isinstance(a.lru_cache.top_k_selector, TokenMaxTopKSelector) == (variant == "quest_oracle")
        outs[variant] = model(out.argmax(-1), 1000).cpu()
        assert torch.isfinite(outs[variant]).all()
    assert (outs["dram"] - outs["quest"]).abs().max().item() > 1e-4 * scale
    with pytest.raises(AssertionError):
        small_args(torch.float32, attention_variant="sparse")


def test_recall_harness_on_a_checkpoint_directory(tmp_path):
    """The evaluation driver end to end on a small random checkpoint written the way
    the Llama-3 download lays it out (params.json + consolidated.00.pth): the loaded
    model decodes the token sequence the CPU restatement of the driver decodes from
    the same weights (page-aligned prefill of 992 of 1003 prefix tokens, 11 + 9 forced
    prompt tokens, then free running), for the paged model and, against the restatement
    with a cache that holds everything, for the full-attention variant; then two
    generated key-value items through tokenizer, model, answer extraction and results
    file."""
    import json

    from dram_attention_amd import LRUCache
    from dram_attention_amd import evaluate as E

    tok = E.ByteTokenizer()
    params = dict(dim=256, n_layers=2, n_heads=8, n_kv_heads=2, vocab_size=tok.n_words,
                  multiple_of=32, ffn_dim_multiplier=1.3, norm_eps=1e-5, rope_theta=500000.0,
                  use_scaled_rope=True)
    cache = dict(lru_hbm_cache_size=256, cache_top_k=128, cache_page_size=16,
                 local_cache_size=128 + 64, max_output_length=64, max_seq_len=1100)
    donor = build(L.ModelArgs(dtype=torch.float32, **params, **cache), 7)
    (tmp_path / "params.json").write_text(json.dumps(params))
    weights = {k: v.detach().cpu() for k, v in donor.named_parameters()}
    weights["rope.freqs"] = torch.zeros(16)         # older checkpoints carry the rope table
    torch.save(weights, tmp_path / "consolidated.00.pth")

    g = torch.Generator().manual_seed(11)
    prefix = torch.randint(0, 256, (1003,), generator=g).tolist()
    suffix = torch.randint(0, 256, (9,), generator=g).tolist()
    for variant, oracle_cache in (("dram", 256), ("full", 1100)):
        model = E.load_model(str(tmp_path), 1100, variant=variant, top_k=128, page_size=16,
                             local_attn_window=128, local_margin=64, lru_hbm_cache_size=256,
                             max_output_length=64, dtype=torch.float32)
        assert model.params.local_cache_size == 128 + 64 and model.params.cache_top_k == 128
        for (name, p), (_, q) in zip(model.named_parameters(), donor.named_parameters()):
            assert torch.equal(p, q), name
        got = E.generate(model, prefix, suffix, 24, page_size=16, stop_tokens=tok.stop_tokens,
                         special_start=tok.special_start)
        args = L.ModelArgs(dtype=torch.float32, **params, **dict(cache, lru_hbm_cache_size=oracle_cache))
        want = M.greedy_generate(M.LlamaOracle(args, donor.state_dict()), prefix, suffix, 24, 16,
                                 tok.stop_tokens, tok.special_start)
        assert got == want and 1 <= len(got) <= 23, (variant, got, want)
        a = model.layers[0].attention.dram_attention
        assert a.dram_kv_cache_size == 816 and isinstance(a.lru_cache, LRUCache) == (variant == "dram")

    # the question line is ~100 byte tokens: they, the completion and the tokens behind the
    # last whole page of the prefix all land in the local cache's room for new rows
    model = E.load_model(str(tmp_path), 1100, top_k=128, page_size=16, local_attn_window=128,
                         local_margin=64, lru_hbm_cache_size=256, max_output_length=192,
                         dtype=torch.float32)
    items = E.synthetic_niah(2, 14, seed=3)
    path = tmp_path / E.results_file_name(1100, "smoke")
    recall = E.evaluate_items(model, tok, items, page_size=16, results_path=str(path), max_gen_len=8)
    rows = [json.loads(line) for line in path.read_text().splitlines()]
    assert [r["index"] for r in rows] == [0, 1] and all(r["recall"] in (0, 1) for r in rows)
    assert recall == sum(r["recall"] for r in rows) / 2
    assert "1100 |" in E.report(str(tmp_path))
    del weights["norm.weight"]
    torch.save(weights, tmp_path / "consolidated.00.pth")
    with pytest.raises(KeyError, match="norm.weight"):
        E.load_model(str(tmp_path), 1100, dtype=torch.float32)
    (tmp_path / "params.json").write_text(json.dumps(dict(params, hidden=3)))
    with pytest.raises(ValueError, match="hidden"):
        E.load_model(str(tmp_path), 1100)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,dim", [(1, 8), (3, 256), (5, 1024), (4, 1032), (7, 4096), (2, 4104), (3, 8192)])
def test_norm_and_swiglu_kernels_match_torch(rows, dim, dtype):
    """The row kernels at the edges of their widths (a wave's rows, a block's, two, four and
    eight vectors a lane) against the torch operators in the CPU branch of the same modules.
    Bound: fp32 sums in another order may turn either of two roundings to the type, each by
    one unit in the last place (up to 2^-7 of the value in bf16, 2^-10 in fp16)."""
    tol = {torch.bfloat16: 2.0 ** -6, torch.float16: 2.0 ** -9, torch.float32: 3e-6}[dtype]
    g = torch.Generator().manual_seed(rows * dim)
    x, y = (torch.randn(1, rows, dim, generator=g).to(dtype) for _ in range(2))
    norm = L.RMSNorm(dim, eps=1e-5).to(dtype)
    with torch.no_grad():
        norm.weight.copy_(1 + 0.1 * torch.randn(dim, generator=g))
        want = norm(x)
        want_sum_norm, want_sum = norm.after_add(x, y)
        gate, up = x * 3, y * 2
        want_glu = torch.nn.functional.silu(gate) * up
        norm = norm.cuda()
        assert L.K.takes(x.cuda(), norm.weight) and L.K.norm_fits(x, norm.weight)   # no fallback
        got = norm(x.cuda())
        got_norm, got_sum = norm.after_add(x.cuda(), y.cuda())
        got_glu = L.K.swiglu_(gate.cuda(), up.cuda())
    assert torch.equal(got_sum.cpu(), want_sum)
    for a, b in ((got, want), (got_norm, want_sum_norm), (got_glu, want_glu)):
        assert torch.allclose(a.cpu().float(), b.float(), rtol=tol, atol=tol * 1e-2)


@pytest.mark.parametrize("dim", [64, 256, 1024, 4096, 8192])
def test_fp32_norm_is_its_roundings_from_float64(dim):
    """Roundings of half a unit in the last place at most: 2.3e-8 in the 2-norm for each of the two
    products; 2.7e-8 for the scale and, halved by the root, for the sum of squares, the mean and the
    sum with eps, which all lie about 1 here: 4.9e-8 together, and 4 % for the sum's inner roundings.
    Rows whose mean is zero, overflows or is not a number come out as the torch operators
    give them."""
    g = torch.Generator(device="cuda").manual_seed(dim)
    x = torch.randn(1, 2 ** 24 // dim, dim, device="cuda", generator=g)
    norm = L.RMSNorm(dim, eps=1e-5).cuda()
    with torch.no_grad():
        norm.weight.copy_(1 + 0.1 * torch.randn(dim, device="cuda", generator=g))
        x64 = x.double()
        want = x64 * torch.rsqrt(x64.square().mean(-1, keepdim=True) + 1e-5) * norm.weight.double()
        assert ((norm(x).double() - want).norm() / want.norm()).item() < 5.1e-8
        odd = torch.zeros(1, 5, dim, device="cuda")
        odd[0, 1:, 0] = torch.tensor([1e30, float("inf"), float("nan"), 1e-30])
        for eps in (0.0, 1e-5):
            bare = L.RMSNorm(dim, eps=eps)
            assert torch.allclose(bare.cuda()(odd).cpu(), bare.cpu()(odd.cpu()), rtol=1e-6, equal_nan=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_swiglu_keeps_its_smallest_results(dtype):
    """Gates far below zero, where exp(-x) nears the largest float and its reciprocal leaves
    the normal numbers before the product does, and beyond, in the row kernel and in the one-token
    layer.  Bound: one turn of the rounding to the type; half the type's smallest step."""
    gate = torch.tensor([-60.0, -80.0, -86.5, -87.0, -87.5, -88.0, -88.5, -89.0, -1e4, 0.0, 3.0, 100.0,
                         -1e-3, 1e-3, -20.0, -40.0], dtype=dtype)
    up = torch.linspace(-2, 2, 16).to(dtype)
    want = (torch.nn.functional.silu(gate) * up).double()
    tiny = 2.0 ** -24 if dtype == torch.float16 else 0.0
    got = L.K.swiglu_(gate.cuda(), up.cuda()).cpu().double()
    assert torch.allclose(got, want, rtol=2.0 ** -7, atol=tiny), (got, want)
    norm = L.RMSNorm(8, eps=0.0).cuda().to(dtype)           # of ones: ones
    w1, w3 = (torch.nn.functional.pad(t[:, None], (0, 7)).cuda() for t in (gate, up))
    with torch.no_grad():
        got = L.K.linear_swiglu(torch.ones(1, 1, 8, dtype=dtype, device="cuda"), norm, w1, w3).flatten().cpu().double()
    assert torch.allclose(got, want, rtol=2.0 ** -7, atol=tiny), (got, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("S,Hq,Hkv,D", [(1, 4, 1, 128), (3, 8, 2, 64), (17, 6, 3, 16)])
def test_rope_kernel_matches_torch(S, Hq, Hkv, D, dtype):
    """In-place rotation of queries and keys against apply_rope on the CPU: fp32 products
    that may be fused, which may turn one rounding to the type by a unit in the last place."""
    g = torch.Generator().manual_seed(S)
    xq, xk = torch.randn(1, S, Hq, D, generator=g).to(dtype), torch.randn(1, S, Hkv, D, generator=g).to(dtype)
    rows = L.rope_table(D, 50, 1e4, True)[11:11 + S]
    q, k = xq.cuda(), xk.cuda()
    L.K.rope_(q, k, rows.cuda())
    tol = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 1e-6}[dtype]
    for got, x in ((q, xq), (k, xk)):
        want = L.apply_rope(x, rows).float()
        assert torch.allclose(got.cpu().float(), want, rtol=tol, atol=tol * 4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dim,n", [(8, 1), (256, 2), (520, 7), (2048, 66), (2056, 33), (4096, 257), (30720, 5),
                                   (136, 8201), (30720, 4099)])
def test_one_token_linear_kernels_match_torch(dim, n, dtype):
    """The one-token layers at the edges of a wave's step (512 elements of 16 bits), of its
    unrolled steps (2048) and at the longest row, odd and single output rows, more pairs of rows than the
    grid has waves (4096, or 2048 where two workgroups' rows fill a unit's LDS), against fp64
    products of the same inputs.  Bound: sums of `dim` fp32 terms, then one turn of each
    rounding to the type (a unit in the last place: 2^-7 of the value in bf16, 2^-10 in
    fp16); silu and the product add one more each."""
    if dim * (4 if dtype == torch.float32 else 2) > L.K.MAX_LINEAR_ROW:
        dim //= 2
    ulp = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 4e-6}[dtype]
    g = torch.Generator().manual_seed(dim + n)

    def draw(*shape, scale=1.0):
        return (scale * torch.randn(*shape, generator=g)).to(dtype).cuda()

    x, res = draw(1, 1, dim), draw(1, 1, n)
    w, w3 = draw(n, dim, scale=dim ** -0.5), draw(n, dim, scale=dim ** -0.5)
    norm = L.RMSNorm(dim).cuda().to(dtype)
    with torch.no_grad():
        norm.weight.copy_(draw(dim, scale=0.1) + 1)
        xn = norm(x).double()

        def rounded(t):
            return t.to(dtype).double()

        def near(got, want, ulps):
            assert torch.allclose(got.double().flatten(), want.flatten(), rtol=ulps * ulp, atol=ulps * ulp * 0.3)

        y, y3 = rounded(xn.flatten() @ w.double().t().contiguous()), rounded(xn.flatten() @ w3.double().t().contiguous())
        near(L.K.linear_logits(x, norm, w), y, 2)
        near(L.K.linear_swiglu(x, norm, w, w3), rounded(torch.nn.functional.silu(y)) * y3, 4)
        near(L.K.linear_add(x, w, res), res.double().flatten() + rounded(x.double().flatten() @ w.double().t().contiguous()), 3)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("Hq,Hkv,D,dim", [(6, 2, 64, 264),
                                          (72, 8, 128, 136)])   # waves go on in each of the three matrices
def test_one_token_qkv_kernel_matches_the_modules(Hq, Hkv, D, dim, dtype):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(1, 1, dim, generator=g).to(dtype).cuda()
    wq, wk, wv = ((torch.randn(h * D, dim, generator=g) / 16).to(dtype).cuda() for h in (Hq, Hkv, Hkv))
    row = L.rope_table(D, 20, 1e4, False, device="cuda")[13:14]
    norm = L.RMSNorm(dim).cuda().to(dtype)
    with torch.no_grad():
        q, k, v = L.K.linear_qkv_rope(x, norm, wq, wk, wv, Hq, Hkv, D, row)
        xn = norm(x)
        # one turn of the projection's rounding, spread over a pair by the rotation, one of the last
        ulp = {torch.bfloat16: 2.0 ** -6, torch.float16: 2.0 ** -9, torch.float32: 4e-6}[dtype]
        for got, w, h, rotated in ((q, wq, Hq, True), (k, wk, Hkv, True), (v, wv, Hkv, False)):
            y = (xn.double() @ w.double().t().contiguous()).to(dtype).view(1, 1, h, D)
            want = L.apply_rope(y, row) if rotated else y
            assert got.shape == want.shape
            assert torch.allclose(got.double(), want.double(), rtol=ulp, atol=ulp)


@pytest.mark.parametrize("n", [1, 3, 4, 4095, 16384, 16385, 128256])
def test_argmax_kernel(n):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randint(-50, 50, (n,), generator=g, device="cuda").float() / 7      # many ties
    token = torch.zeros(1, dtype=torch.int64, device="cuda")

    def check():
        L.K.argmax_into(x, token)
        best = float("nan") if x.isnan().any() else x.max().item()
        hits = (x.isnan() if best != best else x == best).nonzero()
        assert token.item() == hits[0].item()

    check()
    x[n // 2] = float("inf")
    check()
    x[n - 1] = float("nan")
    check()
    x.fill_(float("-inf"))
    check()


def test_greedy_decoding_chooses_by_the_argmax_kernel_in_any_grad_mode(monkeypatch):
    args = small_args(torch.bfloat16)
    calls, argmax_into = [], L.K.argmax_into
    monkeypatch.setattr(L.K, "argmax_into", lambda logits, token: calls.append(1) or argmax_into(logits, token))
    for grad in (True, False):
        model = build(args, 13)
        model(torch.arange(600, device="cuda")[None] % args.vocab_size, 0)
        calls.clear()
        with torch.set_grad_enabled(grad):
            dec = L.GraphedDecoder(model, 600, 5)
            for _ in range(3):
                logits = dec.step()
                assert dec.token.item() == logits.argmax(-1).item() and not logits.requires_grad
        assert len(calls) == 2          # the eager step and the captured one


def test_greedy_decoding_writes_no_further_than_its_token():
    """A caller's token of another type (int32 is one that embeddings take) is written by torch: the
    arg-max kernel writes eight bytes."""
    args = small_args(torch.bfloat16)
    model = build(args, 12)
    model(torch.arange(600, device="cuda")[None] % args.vocab_size, 0)
    dec = L.GraphedDecoder(model, 600, 5)
    around = torch.full((4,), -7, dtype=torch.int32, device="cuda")
    around[1] = 5
    dec.token = around[1:2].view(1, 1)
    with torch.no_grad():
        for _ in range(4):              # eager, captured, replayed
            logits = dec.step()
            assert around.tolist() == [-7, logits.argmax(-1).item(), -7, -7]


def test_a_hooked_or_replaced_module_is_still_called():
    """The one-token kernels leave out no module that somebody watches or has exchanged."""
    args = small_args(torch.bfloat16)
    model = build(args, 8)
    prompt = torch.arange(600, device="cuda")[None] % args.vocab_size
    model(prompt, 0)
    seen = []
    block = model.layers[1]
    handles = [m.register_forward_hook(lambda mod, inp, out: seen.append(mod))
               for m in (block.attention, block.feed_forward.w1, block.ffn_norm, model.output)]
    token = torch.tensor([[5]], device="cuda")
    model(token, 600)
    assert set(seen) == {block.attention, block.feed_forward.w1, block.ffn_norm, model.output} and len(seen) == 4
    for h in handles:
        h.remove()

    class Doubled(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner, self.calls = inner, 0

        def forward(self, x):
            self.calls += 1
            return 2 * self.inner(x)

    block.attention.wo = Doubled(block.attention.wo)
    model(token, 601)
    assert block.attention.wo.calls == 1
    # shapes that do not belong together are torch's to refuse, as before
    model.layers[0].attention.wk = torch.nn.Linear(args.dim, 8, bias=False, device="cuda", dtype=args.dtype)
    with pytest.raises(RuntimeError):
        model(token, 602)
    with pytest.raises(RuntimeError), torch.no_grad():
        L.RMSNorm(64).cuda()(torch.randn(2, 32, device="cuda"))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_block_tail_kernel_equals_its_three_parts(dtype):
    g = torch.Generator(device="cuda").manual_seed(9)

    def draw(*shape):
        return (torch.randn(*shape, device="cuda", generator=g) / 8).to(dtype)

    dim, attn, hidden = 264, 384, 520
    x, att = draw(1, 1, dim), draw(1, 1, 6, 64)
    wo, w1, w3, w2 = draw(dim, attn), draw(hidden, dim), draw(hidden, dim), draw(dim, hidden)
    norm = L.RMSNorm(dim).cuda().to(dtype)
    with torch.no_grad():
        h = L.K.linear_add(att, wo, x)
        want = L.K.linear_add(L.K.linear_swiglu(h, norm, w1, w3), w2, h)
        assert torch.equal(L.K.block_tail(att, wo, x, norm, w1, w3, w2), want)


@pytest.mark.parametrize("length", [1, 600])
def test_a_watched_projection_keeps_its_output(length):
    """What a forward hook keeps of a projection is what the projection returned: rotation
    and SwiGLU work in place only on outputs that nobody else holds."""
    args = small_args(torch.bfloat16)
    model = build(args, 9)
    model(torch.arange(600, device="cuda")[None] % args.vocab_size, 0)
    a, f = model.layers[0].attention, model.layers[0].feed_forward
    kept = {}
    for name, m in (("wq", a.wq), ("wk", a.wk), ("w1", f.w1)):
        m.register_forward_hook(lambda mod, inp, out, name=name: kept.__setitem__(name, (inp[0], out)))
    tokens = torch.arange(length, device="cuda")[None] % args.vocab_size
    model(tokens, 600 if length == 1 else 0)
    for name, (x, out) in kept.items():
        assert torch.equal(torch.nn.functional.linear(x, dict(wq=a.wq, wk=a.wk, w1=f.w1)[name].weight), out), name


def test_an_instance_forward_is_still_called():
    args = small_args(torch.bfloat16)
    model = build(args, 10)
    model(torch.arange(600, device="cuda")[None] % args.vocab_size, 0)
    calls, w2 = [], model.layers[1].feed_forward.w2
    inner = w2.forward
    w2.forward = lambda x: (calls.append(1), inner(x))[1]
    model(torch.tensor([[5]], device="cuda"), 600)
    assert calls == [1]


def test_a_function_mode_sees_the_operators_of_a_token():
    """What a mode that counts calls sees of a decode step: the projections of every layer."""
    from torch.overrides import TorchFunctionMode

    class Count(TorchFunctionMode):
        linears = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.linears += func is torch.nn.functional.linear
            return func(*args, **(kwargs or {}))

    args = small_args(torch.bfloat16)
    model = build(args, 15)
    model(torch.arange(600, device="cuda")[None] % args.vocab_size, 0)
    with Count() as count:
        model(torch.tensor([[5]], device="cuda"), 600)
    assert count.linears == 7 * args.n_layers + 1


def test_rotation_takes_a_table_that_starts_anywhere():
    """Rows of a table four bytes off the kernels' alignment: torch's operators, the same values but
    for products that may be fused (a turn of the rounding: 2^-7)."""
    args = small_args(torch.bfloat16)
    attention = build(args, 16).layers[0].attention
    seen = []
    attention.dram_attention.register_forward_pre_hook(lambda mod, inp: seen.append(inp))
    x = torch.randn(1, 200, args.dim, device="cuda", dtype=torch.bfloat16,
                    generator=torch.Generator(device="cuda").manual_seed(1))
    rows = L.rope_table(attention.head_dim, 200, 1e4, False, device="cuda")
    odd = torch.empty(rows.numel() + 1, device="cuda")[1:].view(rows.shape).copy_(rows)
    with torch.no_grad():
        attention(x, 0, rows)
        attention(x, 0, odd)
    for a, b in zip(*seen):
        assert torch.allclose(a.float(), b.float(), rtol=2.0 ** -7, atol=2.0 ** -9)


@pytest.mark.parametrize("n", [8, 2056, 100000])
def test_swiglu_in_place_of_either_operand(n):
    from dram_attention_amd import _lib

    g = torch.Generator(device="cuda").manual_seed(n)
    gate, up = (torch.randn(n, device="cuda", generator=g).bfloat16() for _ in range(2))
    results = []
    for place in (None, 0, 1):
        operands = [gate.clone(), up.clone()]
        out = torch.empty_like(gate) if place is None else operands[place]
        _lib.check(_lib.load().da_swiglu(operands[0].data_ptr(), operands[1].data_ptr(), out.data_ptr(), n,
                                         _lib.dtype_code(gate.dtype), _lib.stream_ptr(gate.device)), "da_swiglu")
        results.append(out)
    assert torch.equal(results[0], results[1]) and torch.equal(results[0], results[2])


def test_norm_and_feed_forward_compile_as_one_graph():
    args = small_args(torch.float32)
    block = build(args, 14).layers[0]
    g = torch.Generator(device="cuda").manual_seed(2)
    x, y = (torch.randn(1, 5, args.dim, device="cuda", generator=g) for _ in range(2))

    def f(x, y):
        normed, total = block.ffn_norm.after_add(x, y)
        return total + block.feed_forward(block.attention_norm(normed))

    with torch.no_grad():
        assert torch.allclose(torch.compile(f, fullgraph=True, backend="eager")(x, y), f(x, y), atol=1e-5, rtol=1e-5)


def test_a_hook_may_exchange_the_attention_output_of_a_token():
    """What a forward hook (or an attention module of another kind) returns reaches the
    projection as any tensor reaches it: strided and broadcast outputs with their own values, another type
    or size refused.  Against the same call with a feed-forward that is watched, which leaves the
    one-token kernels out: one turn of a rounding to the type here or there, 2^-6 of the largest logit."""
    args = small_args(torch.bfloat16)
    token = torch.tensor([[5]], device="cuda")
    prompt = torch.arange(600, device="cuda")[None] % args.vocab_size

    def strided(out):
        wide = torch.full((*out.shape[:-1], 2 * out.shape[-1]), 7.0, dtype=out.dtype, device="cuda")
        wide[..., ::2] = out
        return wide[..., ::2]

    def run(change, watched):
        model = build(args, 11)
        model(prompt, 0)
        block = model.layers[1]
        if watched:
            block.feed_forward.register_forward_hook(lambda mod, inp, out: None)
        block.attention.dram_attention.register_forward_hook(lambda mod, inp, out: change(out))
        return model(token, 600)

    for change in (strided, lambda out: out.new_ones(()).expand_as(out), lambda out: out.transpose(2, 3),
                   lambda out: torch.nn.Parameter(out.flatten()[1:].new_zeros(out.numel() + 1)[1:].view_as(out))):
        got, want = run(change, False), run(change, True)
        assert (got - want).abs().max() <= 2.0 ** -6 * want.abs().max()
    for change in (lambda out: out.float(), lambda out: out[:, :, :-1], lambda out: out.cpu()):
        for watched in (False, True):
            with pytest.raises(RuntimeError):
                run(change, watched)


def test_transforms_see_the_norm_as_torch_operators():
    """vmap, forward-mode derivatives and tracing, which no_grad leaves on, get torch's
    operators, so that what they compute is not lost."""
    from torch.autograd import forward_ad

    norm = L.RMSNorm(64).cuda()
    x, t = torch.randn(2, 3, 64, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).unbind(0)
    with torch.no_grad():
        want = norm(x)
        assert torch.allclose(torch.vmap(norm)(x), want, atol=1e-6)
        with forward_ad.dual_level():
            tangent = forward_ad.unpack_dual(norm(forward_ad.make_dual(x, t))).tangent
        assert tangent is not None and torch.isfinite(tangent).all() and tangent.abs().max() > 0
        traced = torch.jit.trace(norm, (x,), check_trace=False)
        assert torch.allclose(traced(t), norm(t), atol=1e-6)


def test_a_rotation_table_of_a_class_of_its_own_is_left_to_the_modules(monkeypatch):
    """A token through a model whose table is a subclass of Tensor: the bits of the modules one by one."""
    class Table(torch.Tensor):
        pass

    args = small_args(torch.bfloat16)
    model, ref = (build(args, 5) for _ in range(2))
    prompt = torch.arange(600, device="cuda")[None] % args.vocab_size
    for m in (model, ref):
        m(prompt, 0)
    model.rope = model.rope.as_subclass(Table)
    got = model(prompt[:, :1], 600)
    with monkeypatch.context() as patch:
        patch.setattr(L.TransformerBlock, "_one_token_kernels", staticmethod(lambda *a: None))
        assert torch.equal(got, ref(prompt[:, :1], 600))
