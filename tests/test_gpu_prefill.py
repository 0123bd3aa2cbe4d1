"""The prefill stage: causal attention over the prompt (reference
dram_attention/dram_attention.py:136, flash_attn_func(causal=True)).

The reference's own test of this stage checks the output's shape only
(dram_attention_test.py:31-60), and flash-attn is a third-party library that is not
here, so the values are held against the closed form: a dense fp32 causal softmax
over the same bf16/fp16 inputs, within atol 2e-2 / rtol 1e-2 (the tolerance of the
attention contract), through the C ABI (da_prefill_attention) and through
DRAMAttention.forward(stage="prefill") with each of its backends."""

import math

import pytest
import torch

from tests.util import close, same

pytestmark = pytest.mark.gpu
DEV = "cuda"
ATOL, RTOL = 2e-2, 1e-2


def dense_causal(xq, xk, xv, scale=None):
    """fp32 softmax(q k^T * scale + causal mask) v per kv head; returns (out (1,S,Hq,D) fp32,
    lse (Hq,S) fp32)."""
    _, S, Hq, D = xq.shape
    Hkv = xk.shape[2]
    rep = Hq // Hkv
    scale = 1.0 / math.sqrt(D) if scale is None else scale
    out = torch.empty(1, S, Hq, D, dtype=torch.float32, device=xq.device)
    lse = torch.empty(Hq, S, dtype=torch.float32, device=xq.device)
    mask = torch.ones(S, S, dtype=torch.bool, device=xq.device).tril_()
    for h in range(Hkv):
        q = xq[0, :, h * rep:(h + 1) * rep].float().transpose(0, 1)          # (rep, S, D)
        s = torch.matmul(q, xk[0, :, h].float().t()) * scale                  # (rep, S, S)
        s.masked_fill_(~mask, float("-inf"))
        lse[h * rep:(h + 1) * rep] = torch.logsumexp(s, dim=-1)
        o = torch.matmul(torch.softmax(s, dim=-1), xv[0, :, h].float())       # (rep, S, D)
        out[0, :, h * rep:(h + 1) * rep] = o.transpose(0, 1)
    return out, lse


def draw(S, Hq, Hkv, D, dtype, seed, spread=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    xq = (torch.randn(1, S, Hq, D, device=DEV, generator=g) * spread).to(dtype)
    xk = (torch.randn(1, S, Hkv, D, device=DEV, generator=g) * spread).to(dtype)
    xv = torch.randn(1, S, Hkv, D, device=DEV, generator=g).to(dtype)
    return xq, xk, xv


@pytest.mark.parametrize("S,Hq,Hkv,D,dtype", [
    (4096 + 517, 32, 8, 128, torch.bfloat16),     # the layer shape, a ragged length
    (1, 4, 1, 128, torch.bfloat16),
    (5, 8, 2, 128, torch.bfloat16),
    (31, 4, 4, 64, torch.bfloat16),
    (33, 4, 2, 128, torch.float16),
    (63, 2, 2, 128, torch.bfloat16),
    (64, 4, 1, 128, torch.bfloat16),
    (65, 8, 8, 64, torch.float16),
    (127, 3, 1, 128, torch.bfloat16),             # rep 3: one head per workgroup
    (129, 6, 3, 128, torch.bfloat16),             # rep 2
    (200, 8, 1, 64, torch.bfloat16),              # rep 8: two workgroups per row block
    (1000, 16, 2, 128, torch.float16),
    (2048, 8, 2, 64, torch.bfloat16),
])
def test_prefill_attention_matches_dense_causal_softmax(S, Hq, Hkv, D, dtype):
    from dram_attention_amd.dram_attention import prefill_attention

    xq, xk, xv = draw(S, Hq, Hkv, D, dtype, S + Hq)
    lse = torch.empty(Hq, S, dtype=torch.float32, device=DEV)
    out = prefill_attention(xq, xk, xv, lse=lse)
    want, want_lse = dense_causal(xq, xk, xv)
    assert out.shape == xq.shape and out.dtype == dtype
    assert close(out.float(), want, ATOL, RTOL)
    assert close(lse, want_lse, 1e-3, 1e-4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,Hq,Hkv,D", [
    # few workgroups: two groups of waves share the keys of 32, 64 or 128 rows; lengths around
    # their tiles and blocks, down to a second group without a tile
    (1, 4, 1, 128), (32, 4, 1, 128), (33, 4, 1, 64), (64, 8, 2, 64), (65, 4, 1, 128), (97, 6, 3, 64),
    (128, 2, 1, 128), (129, 5, 5, 128), (191, 4, 2, 128), (193, 3, 3, 64), (257, 12, 3, 128), (385, 14, 2, 64),
    (1030, 10, 5, 64),
    # 256 and 258 workgroups at D 128, 360 and 362 at D 64: the last on this side, the first beyond
    (128, 512, 128, 128), (129, 344, 86, 128), (257, 128, 128, 128), (257, 129, 129, 128), (129, 258, 129, 128),
    (128, 720, 180, 64), (65, 724, 181, 64), (257, 180, 180, 64), (300, 181, 181, 64),
])
def test_prefill_attention_on_both_sides_of_the_key_split(S, Hq, Hkv, D, dtype):
    """Peaked scores, so that the groups' maxima differ.  Against the dense fp32 softmax: the
    weights' and the output's rounding, 2^-9 each of the value in bf16 and 2^-12 in fp16, and
    sums of weights near one; the tolerance of the contract covers them, fp16 gets an eighth."""
    from dram_attention_amd.dram_attention import prefill_attention

    xq, xk, xv = draw(S, Hq, Hkv, D, dtype, S + Hq, spread=1.7)
    lse = torch.empty(Hq, S, dtype=torch.float32, device=DEV)
    out = prefill_attention(xq, xk, xv, lse=lse)
    want, want_lse = dense_causal(xq, xk, xv)
    factor = 1.0 if dtype == torch.bfloat16 else 0.125
    assert close(out.float(), want, ATOL * factor, RTOL * factor)
    assert close(lse, want_lse, 1e-3, 1e-4)


def test_prefill_attention_takes_strided_views_and_peaked_scores():
    """Rows taken out of a fused (S, Hq + 2 Hkv, D) projection, and scores spread widely
    enough that the running maximum moves many times."""
    from dram_attention_amd.dram_attention import prefill_attention

    S, Hq, Hkv, D = 777, 8, 2, 128
    g = torch.Generator(device=DEV).manual_seed(3)
    qkv = (torch.randn(1, S, Hq + 2 * Hkv, D, device=DEV, generator=g) * 3.0).bfloat16()
    xq, xk, xv = qkv[:, :, :Hq], qkv[:, :, Hq:Hq + Hkv], qkv[:, :, Hq + Hkv:]
    out = prefill_attention(xq, xk, xv, scale=0.5)
    want, _ = dense_causal(xq, xk, xv, scale=0.5)
    assert close(out.float(), want, ATOL, RTOL)
    # the first row attends to itself only: its output is its value row, exactly
    assert same(out[0, 0].view(Hkv, Hq // Hkv, D), xv[0, 0][:, None].expand(-1, Hq // Hkv, -1))


def test_prefill_attention_at_the_headline_prompt_length_on_sampled_rows():
    """configs[2]'s prompt (135 152 tokens, 32 q / 8 kv heads, D 128, bf16) through the
    kernel once; rows sampled from the first, a middle and the last blocks, and around
    tile boundaries, are held against a dense fp32 causal softmax over all their keys."""
    from dram_attention_amd.dram_attention import prefill_attention

    S, Hq, Hkv, D = 131072 + 4096 - 16, 32, 8, 128
    rep = Hq // Hkv
    xq, xk, xv = draw(S, Hq, Hkv, D, torch.bfloat16, 5)
    lse = torch.empty(Hq, S, dtype=torch.float32, device=DEV)
    out = prefill_attention(xq, xk, xv, lse=lse)
    rows = torch.tensor(sorted(set(
        list(range(0, 70)) + list(range(65500, 65570)) + [4095, 4096, 4097, 100000, 100063, 100064, 131071, 131072]
        + list(range(S - 40, S)))), device=DEV)
    scale = 1.0 / math.sqrt(D)
    for h in range(Hkv):
        q = xq[0, rows, h * rep:(h + 1) * rep].float().transpose(0, 1)       # (rep, R, D)
        s_ = torch.matmul(q, xk[0, :, h].float().t()) * scale                 # (rep, R, S)
        keys = torch.arange(S, device=DEV)
        s_.masked_fill_(keys[None, None, :] > rows[None, :, None], float("-inf"))
        want = torch.matmul(torch.softmax(s_, dim=-1), xv[0, :, h].float()).transpose(0, 1)   # (R, rep, D)
        assert close(out[0, rows, h * rep:(h + 1) * rep].float(), want, ATOL, RTOL)
        assert close(lse[h * rep:(h + 1) * rep][:, rows], torch.logsumexp(s_, dim=-1), 1e-3, 1e-4)
    assert torch.isfinite(out.float()).all()


def test_prefill_attention_rejects_what_the_kernel_does_not_cover():
    from dram_attention_amd.dram_attention import (causal_prefill_attention, prefill_attention,
                                                   prefill_attention_supported)

    xq, xk, xv = draw(16, 4, 2, 128, torch.float32, 0)
    assert not prefill_attention_supported(xq)
    with pytest.raises(RuntimeError, match="head_dim 64 or 128"):
        prefill_attention(xq, xk, xv)
    xq, xk, xv = draw(16, 4, 2, 32, torch.bfloat16, 0)
    with pytest.raises(RuntimeError, match="head_dim 64 or 128"):
        prefill_attention(xq, xk, xv)
    with pytest.raises(RuntimeError, match="Unsupported prefill backend"):
        causal_prefill_attention(xq, xk, xv, backend="triton")
    # "auto" still answers for such shapes, through torch
    xq, xk, xv = draw(100, 4, 2, 32, torch.float32, 1)
    want, _ = dense_causal(xq, xk, xv)
    assert close(causal_prefill_attention(xq, xk, xv), want, 1e-4, 1e-4)


@pytest.mark.parametrize("backend", ["native", "sdpa", "blocked", "auto"])
def test_module_prefill_stage_values_at_the_layer_shape(backend):
    """DRAMAttention.forward(stage="prefill") at bf16, 32 q / 8 kv heads, D 128, a length
    that is no multiple of the block sizes: the returned output against the dense fp32
    causal softmax, with every backend the module can attend with."""
    from dram_attention_amd import DRAMAttention, LRUCache

    S = 4096 + 517
    xq, xk, xv = draw(S, 32, 8, 128, torch.bfloat16, 11)
    m = DRAMAttention(max_output_length=4, lru_hbm_cache_size=1024, local_cache_size=512,
                      page_size=16, top_k=256, n_kv_heads=8, head_dim=128, device=DEV)
    m.prefill_backend = backend
    try:
        out = m(xq, xk, xv, start_pos=0, stage="prefill")
    except RuntimeError as exc:
        if backend == "sdpa":
            pytest.skip(f"torch's fused attention refuses this shape here: {exc}")
        raise
    want, _ = dense_causal(xq, xk, xv)
    assert out.shape == xq.shape and out.dtype == torch.bfloat16
    assert close(out.float(), want, ATOL, RTOL)
    assert isinstance(m.lru_cache, LRUCache) and m.dram_kv_cache_size == (S - 512 + 16) // 16 * 16


def _plain_prefill(xq, xk, xv):
    """da_prefill_attention_f32 itself, whatever the length."""
    from dram_attention_amd import _lib

    S, Hq, D = xq.shape[1:]
    out, lse = torch.empty(1, S, Hq, D, device=DEV), torch.empty(Hq, S, device=DEV)
    _lib.check(_lib.load().da_prefill_attention_f32(
        xq.data_ptr(), xq.stride(1), xq.stride(2), xk.data_ptr(), xk.stride(1), xk.stride(2), xv.data_ptr(),
        xv.stride(1), xv.stride(2), S, Hq, xk.shape[2], D, 1 / math.sqrt(D), out.data_ptr(), out.stride(1),
        out.stride(2), lse.data_ptr(), _lib.stream_ptr(xq.device)), "plain")
    return out, lse


def _split_prefill(xq, xk, xv):
    """da_prefill_attention_f32_split itself, whatever the length, in a workspace of NaN bytes."""
    from dram_attention_amd import _lib

    S, Hq, D = xq.shape[1:]
    Hkv = xk.shape[2]
    out, lse = torch.empty(1, S, Hq, D, device=DEV), torch.empty(Hq, S, device=DEV)
    room = torch.full((4096 + -(-S // 64) * Hkv * 768 * D,), 255, dtype=torch.uint8, device=DEV)
    _lib.check(_lib.load().da_prefill_attention_f32_split(
        xq.data_ptr(), xq.stride(1), xq.stride(2), xk.data_ptr(), xk.stride(1), xk.stride(2), xv.data_ptr(),
        xv.stride(1), xv.stride(2), S, Hq, Hkv, D, 1 / math.sqrt(D), out.data_ptr(), out.stride(1), out.stride(2),
        lse.data_ptr(), room.data_ptr(), room.numel(), _lib.stream_ptr(xq.device)), "split")
    return out, lse


@pytest.mark.parametrize("S,Hq,Hkv,D", [
    (1, 4, 1, 64), (15, 8, 2, 64), (16, 4, 4, 128), (17, 6, 3, 64), (31, 2, 1, 128), (32, 3, 1, 64),
    (33, 8, 1, 128), (63, 4, 2, 64), (65, 5, 5, 128), (1000, 8, 2, 64), (2049, 12, 3, 128),
])
def test_fp32_prefill_kernel_matches_dense_float64(S, Hq, Hkv, D):
    """The fp32 kernel at the edges of its tiles (16 rows, 32 keys), every grouping of
    heads and both head sizes, on rows cut out of a wider projection.  Bound: products and
    sums of fp32, i.e. score errors of about sqrt(D) 2^-24 times the scores' size (|s| up to ~10 here),
    which the exponential turns into relative errors of the weights: 1e-5."""
    from dram_attention_amd.dram_attention import (causal_prefill_attention, prefill_attention_f32,
                                                   prefill_attention_f32_supported)

    g = torch.Generator(device=DEV).manual_seed(S)
    qkv = torch.randn(1, S, Hq + 2 * Hkv, D, device=DEV, generator=g) * 1.5
    xq, xk, xv = qkv[:, :, :Hq], qkv[:, :, Hq:Hq + Hkv], qkv[:, :, Hq + Hkv:]
    assert prefill_attention_f32_supported(xq, xk, xv)
    lse = torch.empty(Hq, S, dtype=torch.float32, device=DEV)
    out = prefill_attention_f32(xq, xk, xv, lse=lse)
    assert same(causal_prefill_attention(xq, xk, xv), out)
    plain, plain_lse = _plain_prefill(xq, xk, xv)        # (the longer of these prompts takes the other kernel)
    rep = Hq // Hkv
    mask = torch.ones(S, S, dtype=torch.bool, device=DEV).triu_(1)
    for h in range(Hq):
        q, k, v = xq[0, :, h].double(), xk[0, :, h // rep].double(), xv[0, :, h // rep].double()
        s_ = (q @ k.t().contiguous() / math.sqrt(D)).masked_fill_(mask, float("-inf"))
        want, want_lse = torch.softmax(s_, -1) @ v, torch.logsumexp(s_, -1)
        assert close(out[0, :, h].double(), want, 1e-5, 1e-5) and close(lse[h].double(), want_lse, 1e-5, 1e-5)
        assert close(plain[0, :, h].double(), want, 1e-5, 1e-5) and close(plain_lse[h].double(), want_lse, 1e-5, 1e-5)


@pytest.mark.parametrize("kernel", ["plain", "split"])
@pytest.mark.parametrize("D", [64, 128])
def test_fp32_prefill_sums_are_short_chains(D, kernel):
    """Summands that lose half of what lies below the sum's last place when they are added one
    after the other, seen in the log-sum-exp.  Sum of the weights: one addition to the running sum per tile of
    32 keys (and five in and behind it), half a unit in the last place each, and that of the result
    (9, to 2^-21).  A single score: half the channels in a chain lie a binade below the whole sum and lose
    nothing; the chains' sum, the scale, the product with ln 2 and the two logarithms remain, half a unit each.
    (The kernel on bf16 parts adds to each of two running sums once per 64 keys, and its score is one sum of the
    large products, exact here, and the small ones: within the same bounds.)"""
    prefill = _plain_prefill if kernel == "plain" else _split_prefill
    S = 8192
    odd = 1.0 + 502 * 2.0 ** -23
    q, k, v = torch.zeros(1, S, 4, D, device=DEV), torch.zeros(1, S, 1, D, device=DEV), torch.ones(1, S, 1, D, device=DEV)
    q[..., 0] = 1.0
    k[:, 32:, :, 0] = math.log(odd) * math.sqrt(D)       # the first tile's scores, zero, stay the reference
    _, lse = prefill(q, k, v)
    n = torch.arange(1, S + 1, device=DEV, dtype=torch.float64)
    weight = (k[0, 32, 0, 0].double() / math.sqrt(D)).exp()
    want = (n.clamp(max=32) + (n - 32).clamp(min=0) * weight).log()
    assert (lse.double() - want).abs().max().item() < (S / 32 + 5 + 8) * 2.0 ** -24

    term = 1.0 + 0.49 * D * 2.0 ** -24                   # 0.49 of the last place of sums in D/2 .. D
    k = torch.full((1, 1, 1, D), term, device=DEV)
    _, lse = prefill(torch.ones(1, 1, 4, D, device=DEV), k, v[:, :1].contiguous())
    want = D * k[0, 0, 0, 0].double().item() / math.sqrt(D)
    assert (lse.double() / want - 1).abs().max().item() < 5 * 2.0 ** -24


@pytest.mark.parametrize("S,Hq,Hkv,D", [
    (1, 4, 1, 64), (2, 1, 1, 128), (31, 8, 2, 128), (32, 2, 1, 64), (33, 3, 1, 64), (63, 6, 3, 128), (64, 4, 4, 64),
    (65, 4, 2, 128), (127, 8, 2, 64), (128, 5, 5, 128), (129, 7, 1, 64), (200, 12, 3, 128), (1283, 8, 2, 64),
])
def test_fp32_prefill_in_three_parts_matches_dense_float64(S, Hq, Hkv, D):
    """The kernel on bf16 parts at the edges of its tiles (32 rows, 32 and 64 keys), every grouping of heads
    and both head sizes, on rows cut out of a wider projection.  Bound: that of the fp32 kernel's test (the
    parts are exact, what is left out of a product is a quarter of one fp32 rounding)."""
    g = torch.Generator(device=DEV).manual_seed(S)
    qkv = torch.randn(1, S, Hq + 2 * Hkv, D, device=DEV, generator=g) * 1.5
    xq, xk, xv = qkv[:, :, :Hq], qkv[:, :, Hq:Hq + Hkv], qkv[:, :, Hq + Hkv:]
    out, lse = _split_prefill(xq, xk, xv)
    mask = torch.ones(S, S, dtype=torch.bool, device=DEV).triu_(1)
    for h in range(Hq):
        q, k, v = xq[0, :, h].double(), xk[0, :, h // (Hq // Hkv)].double(), xv[0, :, h // (Hq // Hkv)].double()
        s_ = (q @ k.t().contiguous() / math.sqrt(D)).masked_fill_(mask, float("-inf"))
        assert close(out[0, :, h].double(), torch.softmax(s_, -1) @ v, 1e-5, 1e-5)
        assert close(lse[h].double(), torch.logsumexp(s_, -1), 1e-5, 1e-5)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38, 2.0 ** 61, 1e-35, 1e-42])
def test_fp32_prefill_operands_that_do_not_split(value, D):
    """One element of the queries, keys or values, first or last, outside what three parts stand for: the bits of
    the kernel on fp32 instructions."""
    S, Hq, Hkv = 70, 4, 2
    for which in range(3):
        for at in (0, -1):
            ops = list(draw(S, Hq, Hkv, D, torch.float32, 3))
            ops[which].view(-1)[at] = value
            (out, lse), (want, want_lse) = _split_prefill(*ops), _plain_prefill(*ops)
            assert same(out, want) and same(lse, want_lse)


@pytest.mark.parametrize("which", [0, 1, 2])
def test_fp32_prefill_finds_one_operand_among_all_workgroups(which):
    """As many workgroups split as there are words for them, several passes each; the one element that does not
    split lies in the middle, in a late pass, or at the end."""
    S, H, D = 2560, 28, 64
    ops = list(draw(S, H, H, D, torch.float32, 6))
    flat = ops[which].view(-1)
    clean, _ = _split_prefill(*ops)
    want, _ = _plain_prefill(*ops)
    assert not torch.equal(clean, want)                  # (the two kernels are told apart by their bits)
    for at in (flat.numel() // 2 + 77, flat.numel() - H * D * 40 + 5, flat.numel() - 1):
        kept = flat[at].item()
        flat[at] = 2.0 ** -110
        (out, lse), (want, want_lse) = _split_prefill(*ops), _plain_prefill(*ops)
        flat[at] = kept
        assert same(out, want) and same(lse, want_lse), at


def test_fp32_prefill_without_memory_for_the_parts(monkeypatch):
    """The workspace is refused, and only that: the plain kernel's bits."""
    from dram_attention_amd.dram_attention import prefill_attention_f32

    ops = draw(1500, 4, 2, 64, torch.float32, 8)
    want, _ = _plain_prefill(*ops)
    assert not same(prefill_attention_f32(*ops), want)
    empty, refused = torch.empty, []

    def no_bytes(*args, **kwargs):
        if kwargs.get("dtype") is torch.uint8:
            refused.append(args)
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", no_bytes)
    assert same(prefill_attention_f32(*ops), want) and len(refused) == 1


def test_fp32_prefill_splits_to_the_ends_of_its_range():
    """Values of 2^60 and 2^-100, scores of products of the two: still float64's result to 1e-5."""
    S, D = 40, 64
    xq, xk, xv = (x.clone() for x in draw(S, 2, 1, D, torch.float32, 4))
    xv[0, ::3] *= 2.0 ** 57
    xv[0, 1::3] = 2.0 ** -100
    xq[..., 0], xk[..., 0] = 2.0 ** 60, 2.0 ** -58
    out, _ = _split_prefill(xq, xk, xv)
    mask = torch.ones(S, S, dtype=torch.bool, device=DEV).triu_(1)
    for h in range(2):
        s_ = (xq[0, :, h].double() @ xk[0, :, 0].double().t().contiguous() / math.sqrt(D)).masked_fill_(mask, float("-inf"))
        want = torch.softmax(s_, -1) @ xv[0, :, 0].double()
        assert ((out[0, :, h].double() - want).abs() <= 1e-5 * want.abs().amax(-1, keepdim=True)).all()


@pytest.mark.parametrize("D", [64, 128])
def test_fp32_prefill_small_weights_keep_their_bits(D):
    """Values that read out the weights (key j has a one in channel j and zeros elsewhere), the first of each 32 keys
    of weight 1 and the others of 2^-100 to 2^-123: every one within what fp32 scores give.  A score of
    123 powers of two is off by 123 * 2^-24 for each rounding of the scale (two) and by half its last place, 2^-18,
    where the reference is subtracted, all times ln 2; the division adds 2^-23."""
    S = 64
    q, k, v = torch.zeros(1, S, 1, D, device=DEV), torch.zeros(1, S, 1, D, device=DEV), torch.zeros(1, S, 1, D, device=DEV)
    q[..., 0] = 1.0
    j = torch.arange(S, device=DEV)
    k[0, :, 0, 0] = -math.log(2) * math.sqrt(D) * torch.where(j % 32 == 0, 0.0, 100 + 23 * (j % 32) / 31)
    v[0, j, 0, j] = 1.0
    out, _ = _split_prefill(q, k, v)
    mask = torch.ones(S, S, dtype=torch.bool, device=DEV).triu_(1)
    s_ = (k[0, :, 0, 0].double() / math.sqrt(D)).expand(S, S).masked_fill(mask, float("-inf"))
    want = torch.softmax(s_, -1)
    bound = (2 * 123 * 2.0 ** -24 + 2.0 ** -18) * math.log(2) + 2.0 ** -23
    got = out[0, :, 0, :S].double()
    worst = ((got - want).abs() / want)[~mask].max().item()
    assert worst <= bound and (got[mask] == 0).all()


@pytest.mark.parametrize("dtype,S,Hq,Hkv,D", [
    (torch.bfloat16, 3600, 40, 40, 64),     # 600 pieces: two rounds and a part
    (torch.float16, 2050, 66, 66, 128),     # 594, of 66 heads: the part's last 32 are not all of one row block
    (torch.bfloat16, 6700, 40, 40, 64),     # 1080: four rounds and a part
    (torch.float32, 2560, 28, 28, 64), (torch.float32, 2300, 8, 2, 128),   # 560 and 144
])
def test_prefill_in_the_order_of_parts_of_a_round_covers_every_row(dtype, S, Hq, Hkv, D):
    """All rows of all heads against torch's blocked form in fp32, where the order of the pieces is not longest
    first.  Bounds of the other prefill tests: 2e-2 and 1e-2 in 16 bits, 1e-5 in fp32."""
    from dram_attention_amd.dram_attention import causal_prefill_attention

    xq, xk, xv = draw(S, Hq, Hkv, D, dtype, 5)
    out = causal_prefill_attention(xq, xk, xv)
    want = causal_prefill_attention(xq.float(), xk.float(), xv.float(), "blocked")
    atol, rtol = (1e-5, 1e-5) if dtype == torch.float32 else (2e-2, 1e-2)
    assert close(out, want, atol, rtol)


def test_fp32_prompts_of_other_shapes_are_torchs():
    """Several sequences, and keys that reach beyond the queries (row i looks at keys 0..i), against the
    single-sequence kernel and the blocked form: fp32 both, 1e-5.  Heads that do not split are refused."""
    from dram_attention_amd.dram_attention import causal_prefill_attention, prefill_attention_f32

    parts = [draw(70, 4, 2, 64, torch.float32, seed) for seed in (1, 2)]
    both = causal_prefill_attention(*(torch.cat(t) for t in zip(*parts)))
    for got, (xq, xk, xv) in zip(both, parts):
        assert close(got, prefill_attention_f32(xq, xk, xv)[0], 1e-5, 1e-5)
    xq, xk, xv = parts[0]
    want = causal_prefill_attention(xq[:, :50].contiguous(), xk, xv, "blocked")
    assert close(causal_prefill_attention(xq[:, :50].contiguous(), xk, xv), want, 1e-5, 1e-5)
    assert close(want, prefill_attention_f32(xq, xk, xv)[:, :50], 1e-5, 1e-5)
    with pytest.raises(RuntimeError):
        causal_prefill_attention(xq[:, :, :3].contiguous(), xk, xv)


def test_fp32_prompt_under_autocast_is_torchs():
    """Autocast turns scaled dot products to its type; 2e-2 is that type's tolerance here."""
    from dram_attention_amd.dram_attention import causal_prefill_attention

    xq, xk, xv = draw(300, 4, 4, 64, torch.float32, 1)
    want = causal_prefill_attention(xq, xk, xv)
    assert want.dtype == torch.float32
    with torch.no_grad(), torch.autocast("cuda", torch.bfloat16):
        got = causal_prefill_attention(xq, xk, xv)
    assert got.dtype == torch.bfloat16 and close(got, want, ATOL, RTOL)


@pytest.mark.parametrize("S,Hq,Hkv,D,dtype", [
    (600, 2, 2, 64, torch.bfloat16), (3000, 8, 2, 64, torch.float32), (9000, 32, 8, 128, torch.bfloat16),
    (12345, 64, 8, 128, torch.float16),
])
def test_page_store_written_beside_attention_is_complete_on_return(S, Hq, Hkv, D, dtype):
    """stage="prefill" writes the page store on a stream of its own while attention runs;
    the host finds it complete when the call returns, slots and store equal init_cache's,
    whatever number of workgroups the rule gives (32, the limit, to 2), twice in a row on one
    module with the keys freed right after the call."""
    from dram_attention_amd import DRAMAttention
    from dram_attention_amd.dram_attention import causal_prefill_attention, store_build_blocks

    assert 2 <= store_build_blocks((1, S, Hq, D), (1, S, Hkv, D), dtype) <= 32
    m, ref = (DRAMAttention(max_output_length=4, lru_hbm_cache_size=256, local_cache_size=256, page_size=16,
                            top_k=64, n_kv_heads=Hkv, head_dim=D, device=DEV, dtype=dtype) for _ in range(2))
    for seed in (1, 2):
        xq, xk, xv = draw(S, Hq, Hkv, D, dtype, seed)
        out = m(xq, xk, xv, start_pos=0, stage="prefill")
        store = m.lru_cache.dram_kv_cache.clone()          # read by the host, nothing waited for
        want = causal_prefill_attention(xq, xk, xv)
        ref.init_cache(xk, xv)
        del xk, xv
        junk = torch.full((S, Hkv, 4 * D), 7.0, device=DEV, dtype=dtype)   # takes the freed memory
        assert same(store, ref.lru_cache.dram_kv_cache)
        for name in ("hbm_kv_cache", "dram_page_to_hbm_page_mapping", "hbm_page_to_dram_page_mapping"):
            assert same(getattr(m.lru_cache, name), getattr(ref.lru_cache, name))
        assert same(out, want)
        del junk


def test_a_refused_prompt_leaves_the_layer_as_it_was():
    from dram_attention_amd import DRAMAttention

    m = DRAMAttention(max_output_length=4, lru_hbm_cache_size=256, local_cache_size=256, page_size=16,
                      top_k=64, n_kv_heads=2, head_dim=64, device=DEV, dtype=torch.bfloat16)
    xq, xk, xv = draw(1000, 4, 2, 64, torch.bfloat16, 1)
    m(xq, xk, xv, start_pos=0, stage="prefill")
    cache, paged = m.lru_cache, m.dram_kv_cache_size
    xq, xk, xv = draw(2000, 4, 2, 64, torch.bfloat16, 2)
    with pytest.raises(ValueError):
        m(xq, xk.half(), xv.half(), start_pos=0, stage="prefill")
    with pytest.raises(ValueError):
        m(xq[:, :0], xk, xv, start_pos=0, stage="prefill")
    assert m.lru_cache is cache and m.dram_kv_cache_size == paged


def test_an_init_cache_of_its_own_gets_the_prompt(monkeypatch):
    """In a subclass, on the layer or in the class's place: called once, with the prompt's keys and values."""
    from dram_attention_amd import DRAMAttention

    class Own(DRAMAttention):
        def init_cache(self, k_cache, v_cache):
            given.append((k_cache, v_cache))
            super().init_cache(k_cache, v_cache)

    xq, xk, xv = draw(1000, 4, 2, 64, torch.bfloat16, 1)
    sizes = dict(max_output_length=4, lru_hbm_cache_size=256, local_cache_size=256, page_size=16, top_k=64,
                 n_kv_heads=2, head_dim=64, device=DEV, dtype=torch.bfloat16)
    given, ref = [], DRAMAttention(**sizes)
    want = ref(xq, xk, xv, start_pos=0, stage="prefill")
    for where in ("subclass", "layer", "class"):
        given.clear()
        m = (Own if where == "subclass" else DRAMAttention)(**sizes)
        with monkeypatch.context() as patch:
            if where == "layer":
                inner = m.init_cache
                m.init_cache = lambda k, v: given.append((k, v)) or inner(k, v)
            if where == "class":
                init_cache = DRAMAttention.init_cache
                patch.setattr(DRAMAttention, "init_cache",
                              lambda self, k, v: given.append((k, v)) or init_cache(self, k, v))
            assert same(m(xq, xk, xv, start_pos=0, stage="prefill"), want)
        assert len(given) == 1 and given[0][0] is xk and given[0][1] is xv, where
        assert same(m.lru_cache.dram_kv_cache, ref.lru_cache.dram_kv_cache)


def test_the_old_page_store_outlives_the_launches_that_read_it(monkeypatch):
    """A second prompt on a layer: the first one's store, which the last decode steps read by address,
    is let go only when the host has waited for what was launched."""
    import weakref

    from dram_attention_amd import DRAMAttention, LRUCache

    m = DRAMAttention(max_output_length=4, lru_hbm_cache_size=256, local_cache_size=256, page_size=16,
                      top_k=64, n_kv_heads=2, head_dim=64, device=DEV, dtype=torch.bfloat16)
    xq, xk, xv = draw(1000, 4, 2, 64, torch.bfloat16, 1)
    m(xq, xk, xv, start_pos=0, stage="prefill")
    old, held, finish = weakref.ref(m.lru_cache.dram_kv_cache), [], LRUCache.finish_build
    monkeypatch.setattr(LRUCache, "finish_build", lambda self: finish(self) or held.append(old() is not None))
    m(xq, xk, xv, start_pos=0, stage="prefill")
    assert held == [True] and old() is None


def test_the_host_link_is_timed_while_no_store_is_being_written(monkeypatch):
    """The rate is kept for the whole process: it must not come from copies that shared the link
    with a page store on its way."""
    from dram_attention_amd import DRAMAttention, LRUCache, dram_attention

    being_built, at_timing = [], []
    init, finish = LRUCache.__init__, LRUCache.finish_build
    monkeypatch.setattr(LRUCache, "__init__", lambda self, *a, **kw: being_built.append(1) or init(self, *a, **kw))
    monkeypatch.setattr(LRUCache, "finish_build", lambda self: finish(self) or being_built.clear())
    monkeypatch.setattr(dram_attention, "host_link_gbps", lambda device: at_timing.append(len(being_built)) or 50.0)
    m = DRAMAttention(max_output_length=4, lru_hbm_cache_size=256, local_cache_size=256, page_size=16,
                      top_k=64, n_kv_heads=2, head_dim=64, device=DEV, dtype=torch.bfloat16)
    xq, xk, xv = draw(1000, 4, 2, 64, torch.bfloat16, 1)
    m(xq, xk, xv, start_pos=0, stage="prefill")
    m.init_cache(xk, xv)
    assert at_timing == [0, 0] and m.link_gbps == 0.95 * 50.0


@pytest.mark.parametrize("stage", ["prefill", "init_cache"])
@pytest.mark.parametrize("why", ["unknown selector", "failing selector", "shorter than the window", "values cut short"])
def test_a_prompt_refused_late_leaves_the_layer_decoding_as_before(why, stage, monkeypatch):
    """Refusals behind the construction of the page cache: the layer keeps its cache, prefix length
    and local window, and its next token is that of a layer that never saw the prompt."""
    from dram_attention_amd import DRAMAttention, dram_attention

    m, ref = (DRAMAttention(max_output_length=8, lru_hbm_cache_size=256, local_cache_size=256, page_size=16,
                            top_k=64, n_kv_heads=2, head_dim=64, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    xq, xk, xv = draw(1000, 4, 2, 64, torch.bfloat16, 1)
    m.init_cache(xk, xv)
    ref.init_cache(xk, xv)
    cache = m.lru_cache
    length = {"shorter than the window": 100, "values cut short": 400}.get(why, 2000)
    q, k, v = draw(length, 4, 2, 64, torch.bfloat16, 2)
    if why == "values cut short":       # (a static cache: 160 of its tokens are paged)
        v = v[:, :-8]
    if why == "unknown selector":
        m.page_selector = "none of them"
    if why == "failing selector":
        m.page_selector = "token_max"

        def failing(*args, **kwargs):
            raise RuntimeError("out of memory")

        monkeypatch.setattr(dram_attention, "TokenMaxTopKSelector", failing)
    with pytest.raises((RuntimeError, ValueError)):
        m.init_cache(k, v) if stage == "init_cache" else m(q, k, v, start_pos=0, stage="prefill")
    m.page_selector = "bound"
    assert m.lru_cache is cache and m.dram_kv_cache_size == ref.dram_kv_cache_size
    xq, xk, xv = draw(1, 4, 2, 64, torch.bfloat16, 3)
    assert same(m(xq, xk, xv, start_pos=1000, stage="generate"), ref(xq, xk, xv, start_pos=1000, stage="generate"))
    assert same(m.cache_k, ref.cache_k) and same(m.cache_v, ref.cache_v)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,local,lru,page,kind", [
    (1500, 200, 320, 16, "plain"), (1511, 200, 320, 16, "plain"),    # pages and a window that ends inside one
    (3000, 1000, 640, 32, "view"), (700, 203, 4096, 16, "plain"),    # strided prompt; static prefix
    (150, 160, 4096, 16, "view"), (700, 16, 0, 16, "plain"),         # the window alone, no slots
    (1500, 200, 320, 16, "odd rows"), (1500, 200, 320, 16, "unlike values"),   # left to the launches of their own
])
def test_prompt_caches_in_one_launch_equal_the_separate_ones(dtype, S, local, lru, page, kind, monkeypatch):
    """Summaries, page cache metadata and window, bit for bit, and which prompts the launch is for."""
    from dram_attention_amd import DRAMAttention, LRUCache

    H, D = 3, 64
    g = torch.Generator(device=DEV).manual_seed(S)

    def rand(width):
        return torch.randn(1, S, H, width, device=DEV, generator=g).to(dtype)

    if kind == "plain":
        k, v = rand(D), rand(D)
    elif kind == "view":
        k, v = rand(2 * D)[..., :D], rand(2 * D)[..., D:]
    elif kind == "odd rows":
        k, v = rand(D + 1)[..., :D], rand(D + 1)[..., :D]
    else:
        k, v = rand(D), rand(2 * D)[..., :D]
    launches, fill = [], DRAMAttention._fill_caches
    monkeypatch.setattr(DRAMAttention, "_fill_caches", lambda *a: launches.append(1) or fill(*a))

    def layer():
        m = DRAMAttention(8, lru, local, page, 4 * page, H, D, device=DEV, dtype=dtype)
        m.init_cache(k, v)
        return m

    one = layer()
    assert len(launches) == (kind in ("plain", "view"))
    with monkeypatch.context() as patch:
        patch.setattr(DRAMAttention, "_caches_in_one_launch", lambda *a: False)
        many = layer()
    for name in ("cache_k", "cache_v"):
        assert torch.equal(getattr(one, name), getattr(many, name)), name
    assert type(one.lru_cache) is type(many.lru_cache) and one.dram_kv_cache_size == many.dram_kv_cache_size
    if isinstance(one.lru_cache, LRUCache):
        for name in ("current_step", "page_access_time", "dram_page_to_hbm_page_mapping",
                     "hbm_page_to_dram_page_mapping", "dram_kv_cache", "hbm_kv_cache"):
            assert torch.equal(getattr(one.lru_cache, name), getattr(many.lru_cache, name)), name
        assert torch.equal(one.lru_cache.top_k_selector.chunk_min_max, many.lru_cache.top_k_selector.chunk_min_max)


@pytest.mark.parametrize("what,stage", [
    ("page cache", "init_cache"),       # (a prompt tells its page cache where to write the store, too)
    ("selector", "init_cache"), ("selector", "prefill"),
    ("selector that refuses", "init_cache"), ("selector that refuses", "prefill"),
])
def test_stand_ins_for_the_page_cache_and_its_selector(what, stage, monkeypatch):
    """Classes put in their places with the signatures of the reference's: init_cache calls the page cache
    with its parameters and no others, the page cache its selector; one that refuses the prompt leaves the layer
    as it was."""
    from dram_attention_amd import DRAMAttention, IPUpperboundTopKSelector, LRUCache, dram_attention, lru_cache

    class Cache(LRUCache):
        def __init__(self, k_cache, v_cache, page_size, top_k, lru_hbm_cache_size=None, hbm_kv_cache_fraction=0.2,
                     device="cuda"):
            made.append(self)
            super().__init__(k_cache, v_cache, page_size, top_k, lru_hbm_cache_size, hbm_kv_cache_fraction, device)

    class Selector(IPUpperboundTopKSelector):
        def __init__(self, k_cache, num_pages, device="cuda"):
            made.append(self)
            if what == "selector that refuses":
                raise RuntimeError("not these keys")
            super().__init__(k_cache, num_pages, device)

    made, (q, k, v) = [], draw(1000, 4, 2, 64, torch.bfloat16, 1)
    m, ref = (DRAMAttention(max_output_length=4, lru_hbm_cache_size=256, local_cache_size=256, page_size=16, top_k=64,
                            n_kv_heads=2, head_dim=64, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    m.init_cache(k, v)
    window = m.cache_k.clone(), m.cache_v.clone()
    _, k, v = draw(1100, 4, 2, 64, torch.bfloat16, 2)
    ref.init_cache(k, v)
    if what == "page cache":
        monkeypatch.setattr(dram_attention, "LRUCache", Cache)
    else:
        monkeypatch.setattr(lru_cache, "IPUpperboundTopKSelector", Selector)
    q = draw(1100, 4, 2, 64, torch.bfloat16, 2)[0]
    prompt = (lambda: m.init_cache(k, v)) if stage == "init_cache" else (lambda: m(q, k, v, start_pos=0, stage="prefill"))
    if what == "selector that refuses":
        with pytest.raises(RuntimeError, match="not these keys"):
            prompt()
        assert made and same(m.cache_k, window[0]) and same(m.cache_v, window[1])
        return
    prompt()
    assert len(made) == 1
    assert same(m.cache_k, ref.cache_k) and same(m.cache_v, ref.cache_v)
    assert same(m.lru_cache.top_k_selector.chunk_min_max, ref.lru_cache.top_k_selector.chunk_min_max)
    for name in ("current_step", "page_access_time", "dram_page_to_hbm_page_mapping", "hbm_page_to_dram_page_mapping"):
        assert same(getattr(m.lru_cache, name), getattr(ref.lru_cache, name)), name
