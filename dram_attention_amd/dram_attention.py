"""DRAM Attention: long prefix in pinned host DRAM, hot pages in an HBM LRU,
recent tokens in a local HBM window; decode attends over (resident pages ++
local window ++ new token) in one split-K pass.

Mirrors dram_attention/dram_attention.py of the reference (DRAMAttention
:7-238): constructor, buffers, ``init_cache`` and ``forward(xq, xk, xv, *,
start_pos, stage)`` keep their meaning and error behaviour.
"""

from __future__ import annotations

import ctypes
import math

import torch
import torch.nn.functional as F

from . import _lib
from .lru_cache import DummyCache, LRUCache
from .lru_kernel import GATHER_BLOCKS, gather_attend_supported, host_link_gbps
from .max_ip_kernel import DA_SCORE_ORDERED_BOUNDS, DA_SCORE_ROUND
from .model_kernels import unobserved
from .topk_selector import IPUpperboundTopKSelector, TokenMaxTopKSelector

# da_page_score flags of a step by whether the summaries' bounds are ordered
SCORE_FLAGS = {False: DA_SCORE_ROUND, True: DA_SCORE_ROUND | DA_SCORE_ORDERED_BOUNDS}


class PagedPrefix:
    """Says that the prefix handed to :func:`decode_attention` is the slot array of
    an LRU page cache whose page stream for this step may still be running.

    FIRST attends over the local window and every slot that keeps its page,
    FIRST_MERGE folds those partial results into one (both may run next to the
    stream), SECOND (after the stream has finished) attends over the re-assigned
    slots and writes the output; FIRST | SECOND does everything at once.  With
    STREAM the page stream itself runs inside the launch of the FIRST pass;
    SECOND | MERGE_ALL is the final merge as a call of its own after FIRST (| STREAM)
    without FIRST_MERGE."""

    FIRST, SECOND, FIRST_MERGE, STREAM, MERGE_ALL = 1, 2, 4, 8, 16

    def __init__(self, page_size: int, scratch, current_step: torch.Tensor, phase: int,
                 gather_blocks: int = 0, page_stores=None, link_gbps: float = 0.0,
                 block_gbps: float = 0.0):
        self.page_size = page_size
        self.scratch = scratch
        self.current_step = current_step
        self.phase = phase
        # blocks per kv head of a page stream that attends over the pages it moves
        # (0: the SECOND pass attends over the re-assigned slots)
        self.gather_blocks = gather_blocks
        # STREAM: (dram_kv_cache, its device-visible address, hbm_kv_cache); the page
        # stream then runs inside the launch of the FIRST pass
        self.page_stores = page_stores
        # STREAM: the host link's rate for reads issued by a kernel and the rate at which
        # one workgroup reads HBM, GB/s (0 = the library's defaults); they decide how
        # many workgroups compute the first pass next to a long stream, not what it computes
        self.link_gbps = link_gbps
        self.block_gbps = block_gbps

    def as_struct(self) -> "_lib.PagedOverlap":
        s = self.scratch
        o = _lib.PagedOverlap(
            page_size=self.page_size, phase=self.phase, slot_epoch=s.slot_epoch.data_ptr(),
            slot_epoch_head_stride=s.slot_epoch.stride(0), epoch=self.current_step.data_ptr(),
            miss_slot=s.miss_slot.data_ptr(), miss_count=s.miss_count.data_ptr(),
            miss_capacity=s.miss_slot.shape[1], gather_blocks=self.gather_blocks)
        if self.phase & self.STREAM:
            dram, dram_ptr, hbm = self.page_stores
            esz = dram.element_size()
            o.dram, o.hbm, o.miss_page = dram_ptr, hbm.data_ptr(), s.miss_page.data_ptr()
            o.dram_head_stride_bytes = dram.stride(0) * esz
            o.dram_page_stride_bytes = dram.stride(1) * esz
            o.hbm_head_stride_bytes = hbm.stride(0) * esz
            o.hbm_slot_stride_bytes = hbm.stride(1) * esz
            o.link_gbps, o.block_gbps = self.link_gbps, self.block_gbps
        return o


def attention_workspace(Hq: int, Hkv: int, D: int, dtype: torch.dtype, p_len: int, capacity: int,
                        miss_tokens: int, device) -> torch.Tensor:
    need = _lib.load().da_decode_attention_workspace_bytes(
        Hq, Hkv, D, _lib.dtype_code(dtype), p_len, capacity, miss_tokens)
    if need == 0:
        raise RuntimeError(f"decode attention does not cover head_dim={D} dtype={dtype}")
    return torch.empty((need + 3) // 4, dtype=torch.float32, device=device)


def decode_attention(
    xq: torch.Tensor,
    prefix_k: torch.Tensor,
    prefix_v: torch.Tensor,
    cache_k: torch.Tensor,
    cache_v: torch.Tensor,
    cache_len,
    new_k: torch.Tensor | None,
    new_v: torch.Tensor | None,
    *,
    workspace: torch.Tensor | None = None,
    out: torch.Tensor | None = None,
    lse: torch.Tensor | None = None,
    scale: float | None = None,
    paged: PagedPrefix | None = None,
    cache_len_offset: int = 0,
) -> torch.Tensor:
    """One query token against [prefix ++ cache rows 0..cache_len ++ new token].

    xq (Hq, D); prefix_k/v (Hkv, T, D) views with a dense last axis (T may be 0);
    cache_k/v (capacity, Hkv, D); cache_len an int, or a one-element int32 GPU
    tensor to which ``cache_len_offset`` is added inside the kernel (so a device
    position counter needs no arithmetic launch); new_k/new_v (Hkv, D) are
    appended at row cache_len (or None).
    Returns (Hq, D) in xq.dtype; fills ``lse`` (Hq, fp32) when given.
    With ``paged`` the work is split around a concurrent page stream; the same
    workspace and ``out`` must be passed to every call of the step.
    """
    Hq, D = xq.shape
    Hkv = cache_k.shape[1]
    _lib.require_gpu(xq, "xq")
    lib = _lib.load()
    dt = _lib.dtype_code(xq.dtype)
    p_len = prefix_k.shape[1] if prefix_k is not None else 0
    capacity = cache_k.shape[0]
    if out is None:
        out = torch.empty(Hq, D, dtype=xq.dtype, device=xq.device)
    if workspace is None:
        miss_tokens = paged.scratch.miss_slot.shape[1] * paged.page_size if paged else 0
        workspace = attention_workspace(Hq, Hkv, D, xq.dtype, p_len, capacity, miss_tokens,
                                        xq.device)
    if isinstance(cache_len, torch.Tensor):
        _lib.require_gpu(cache_len, "cache_len")
        if cache_len.dtype != torch.int32:
            raise TypeError("a device-side cache length must be int32")
        len_host, len_dev = int(cache_len_offset), cache_len.data_ptr()
    else:
        len_host, len_dev = int(cache_len), None
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    for t in (xq, prefix_k, prefix_v, cache_k, cache_v, new_k, new_v):
        if t is not None and t.numel() and t.stride(-1) != 1:
            raise ValueError("head_dim must be the dense axis of every operand")
    overlap = paged.as_struct() if paged is not None else None
    _lib.check(
        lib.da_decode_attention_paged(
            xq.data_ptr(), xq.stride(0), Hq, Hkv, D, dt,
            prefix_k.data_ptr() if p_len else None, prefix_v.data_ptr() if p_len else None,
            prefix_k.stride(1) if p_len else 0, prefix_k.stride(0) if p_len else 0, p_len,
            cache_k.data_ptr(), cache_v.data_ptr(), cache_k.stride(0), cache_k.stride(1),
            capacity, len_host, len_dev,
            new_k.data_ptr() if new_k is not None else None,
            new_v.data_ptr() if new_v is not None else None,
            new_k.stride(0) if new_k is not None else 0,
            scale, out.data_ptr(), out.stride(0),
            lse.data_ptr() if lse is not None else None,
            workspace.data_ptr(), workspace.numel() * workspace.element_size(),
            ctypes.byref(overlap) if overlap is not None else None,
            _lib.stream_ptr(xq.device),
        ),
        "da_decode_attention",
    )
    return out


def prefill_attention_supported(xq: torch.Tensor) -> bool:
    """Whether the library's own causal prefill kernel takes this query tensor."""
    return (xq.is_cuda and xq.dtype in (torch.bfloat16, torch.float16)
            and xq.shape[-1] in (64, 128))


def prefill_attention(xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor, *,
                      scale: float | None = None, lse: torch.Tensor | None = None) -> torch.Tensor:
    """Causal attention over the prompt on the library's kernel (da_prefill_attention):
    (1,S,Hq,D), (1,S,Hkv,D) x 2 -> (1,S,Hq,D); fills ``lse`` (Hq, S) fp32 when given.
    Replaces flash_attn_func(xq, xk, xv, causal=True), reference dram_attention.py:136."""
    out, args = _prefill_operands(xq, xk, xv, lse)
    S, Hq, D = xq.shape[1:]
    _lib.check(
        _lib.load().da_prefill_attention(
            *args, S, Hq, xk.shape[2], D, _lib.dtype_code(xq.dtype),
            float(scale) if scale is not None else 1.0 / math.sqrt(D), out.data_ptr(),
            out.stride(1), out.stride(2), lse.data_ptr() if lse is not None else None,
            _lib.stream_ptr(xq.device)),
        "da_prefill_attention")
    return out


def prefill_attention_f32_supported(xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor) -> bool:
    """Whether the library's fp32 prefill kernel takes these tensors as they are (it has no
    backward and no other derivative, so operands that autograd or a transform follows stay
    with torch, as do token strides above the kernel's 2^24 bytes, several sequences, keys of
    another length, and autocast, under which torch attends in the 16-bit type)."""
    q_shape, k_shape = xq.shape, xk.shape
    if not xq.is_cuda or not len(q_shape) == len(k_shape) == 4 or xv.shape != k_shape:
        return False
    (bsz, S, Hq, D), (n_seqs, Skv, Hkv, Dk) = q_shape, k_shape
    if not (bsz == n_seqs == 1 and Skv == S and Dk == D and D in (64, 128) and Hkv > 0 and Hq % Hkv == 0
            and unobserved() and not torch.is_autocast_enabled()):
        return False
    device, grad = xq.device, torch.is_grad_enabled()
    for t in (xq, xk, xv):
        stride = t.stride()
        if (type(t) not in (torch.Tensor, torch.nn.Parameter) or t.dtype is not torch.float32 or t.device != device
                or stride[3] != 1 or stride[1] % 4 or stride[2] % 4 or stride[1] > 1 << 22 or t.data_ptr() % 16
                or (grad and t.requires_grad)):
            return False
    return True


def prefill_attention_f32(xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor, *,
                          scale: float | None = None,
                          lse: torch.Tensor | None = None) -> torch.Tensor:
    """:func:`prefill_attention` for an fp32 layer: fp32 products and sums throughout
    (da_prefill_attention_f32), and for a prompt of some length, where there is memory for its keys
    and values in three bf16 parts each, the products of those parts, which are as exact
    (da_prefill_attention_f32_split)."""
    out, args = _prefill_operands(xq, xk, xv, lse)
    if xq.dtype != torch.float32:
        raise TypeError(f"prefill_attention_f32 takes float32, got {xq.dtype}")
    S, Hq, D = xq.shape[1:]
    lib, Hkv = _lib.load(), xk.shape[2]
    args += (S, Hq, Hkv, D, float(scale) if scale is not None else 1.0 / math.sqrt(D), out.data_ptr(),
             out.stride(1), out.stride(2), lse.data_ptr() if lse is not None else None)
    need = lib.da_prefill_attention_f32_workspace_bytes(S, Hq, Hkv, D)
    if need:
        try:
            room = torch.empty(need, dtype=torch.uint8, device=xq.device)
        except torch.cuda.OutOfMemoryError:
            need = 0
    if need:
        _lib.check(lib.da_prefill_attention_f32_split(*args, room.data_ptr(), need, _lib.stream_ptr(xq.device)),
                   "da_prefill_attention_f32_split")
    else:
        _lib.check(lib.da_prefill_attention_f32(*args, _lib.stream_ptr(xq.device)), "da_prefill_attention_f32")
    return out


def _prefill_operands(xq, xk, xv, lse):
    """Checks of the native prefill kernels; (output, pointer and stride arguments)."""
    bsz, S, Hq, D = xq.shape
    assert bsz == 1, "Only support batch size 1"
    for name, t in (("xq", xq), ("xk", xk), ("xv", xv)):
        _lib.require_gpu(t, name)
        if t.stride(-1) != 1:
            raise ValueError("head_dim must be the dense axis of every operand")
    if xk.shape != xv.shape or xk.shape[1] != S or xk.shape[3] != D or not (
            xq.dtype == xk.dtype == xv.dtype):
        raise ValueError("query, keys and values must agree in length, head size and type")
    if lse is not None and (lse.shape != (Hq, S) or lse.dtype != torch.float32
                            or not lse.is_contiguous()):
        raise ValueError("lse must be a contiguous fp32 tensor of shape (Hq, S)")
    out = torch.empty(1, S, Hq, D, dtype=xq.dtype, device=xq.device)
    return out, (xq.data_ptr(), xq.stride(1), xq.stride(2), xk.data_ptr(), xk.stride(1),
                 xk.stride(2), xv.data_ptr(), xv.stride(1), xv.stride(2))


def store_build_blocks(q_shape, k_shape, dtype: torch.dtype, page_size: int = 16, resident: float = 0.0) -> int:
    """Workgroups that write the page store of the keys (and values) of ``k_shape`` next to prefill attention,
    the share ``resident`` of whose pages go into slots as well.  Each takes a compute unit from it, and
    once the writes fill the link (57 GB/s) every miss of attention's caches waits behind them: up to the count
    ``most`` another workgroup makes the store faster, the next few cost attention a fifth or more.  So up to
    a ratio of the store's time on a full link to attention's there are ``most`` (fewer where the store is far
    shorter), and beyond it, as the end of the store decides, the more the larger the ratio is.  A workgroup
    moves more the larger its pages are, and less beside fp32 attention, beside heads that do not share
    their keys and values, whose attention uses more of the memory, and where its pages go into slots.
    us by workgroups (* the one taken here; pages of 16 tokens, up to 0.4 resident where not stated):

      64/8 heads, D 128 (8 KB) 30455 tokens: 2 14103, 3 13413, *5, 7 13234, 10 13523, 28 14523
      32/8, D 128 20922: 4 3415, 5 3296, *7 3216, 8 3274, 9 3632, 12 3836, 32 4093
        10357: 6 1066, *7 928, 8 934, 10 1209, 16 1212; 6784: 6 696, *7 633, 8 654, 10 676, 12 630, 16 689, 32 705
        4910: 7 459, 8 483, 12 447, *16 447, 20 440, 24 445, 32 455; 2778: 8 350, 16 322, 24 307, *32 305
      40/10, D 128, 0.9 resident 20545: 5 4323, 7 4061, 8 4011, *9, 10 3981, 14 4778
      16/16, D 128 39023: 6 8325, 7 7144, *8 6144, 9 7223, 12 8664; 20677: 8 3353, 12 3517, 14 3377, *16 3403, 32 3736
      16/16, D 64 (4 KB) 30548: 8 3347, 9 3011, *10 2757, 12 3134, 16 3124; 15292: 10 1391, 16 1474, *24 1335, 32 1305
        all resident 39957: 7 6258, 10 4708, 12 4046, *13, 14 4014, 20 5016
      32/8, D 128, fp32 (16 KB) 3370: 5 676, *6 660, 7 712, 8 763, 12 766, 32 898; 1888: 6 398, 8 411, *12 375, 16 382

    Over 306 prompts of 29 layouts (heads, type, page) that is 1.3 % slower on average than the best of 13 to 16
    counts, and 11 % at most: 5265 tokens of 24/8 heads, D 128, fp32, *6 1072, 5 969.  Over 140 drawn ones, up to all
    resident, 0.9 % and 10 %.  (One count two or three off costs 15 to 30 % at the worst places.)"""
    _, S, Hq, D = q_shape
    Hkv = k_shape[2]
    f32, shared = dtype == torch.float32, Hq >= 3 * Hkv
    flops_per_s, esize = (1.9e14, 4) if f32 else (1e15, 2)
    attention_s = max(1e-9, 2.0 * S * S * Hq * D / flops_per_s)    # (no queries: attention refuses them)
    store_s = 2e-5 + 2.0 * k_shape[1] * Hkv * D * esize / 57e9    # (20 us until the first pages are across)
    ratio, page_bytes = store_s / attention_s, page_size * 2 * D * esize
    if page_bytes >= 16384:
        most, line, least, slope = 6, 1.3 if shared else 1.5, 12, 4.0
    elif page_bytes >= 8192:
        most, line, least, slope = 8 - shared + f32, 1.2 if shared else 1.45, 14, 5.5
    else:
        most, line, least, slope = 10, 1.1 if shared else 1.4, 20, 5.5
    if ratio < line:
        most = int(most * (1 + (0.2 if f32 or page_bytes >= 16384 else 0.4) * resident))
        return max(2, min(most, math.ceil(30 * ratio)))
    return min(32, max(least, 2 * int(slope * ratio)))


_build_streams = {}


def build_stream(device: torch.device) -> torch.cuda.Stream:
    """The stream that page stores are written on next to prefill attention: one per device
    for all layers (what it is given waits for its caller's stream and is waited for before
    the call returns; a stream of its own would cost every new layer's first prompt
    another 0.2 ms)."""
    stream = _build_streams.get(device)
    if stream is None:
        stream = _build_streams.setdefault(device, torch.cuda.Stream(device=device))
    return stream


def causal_prefill_attention(xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor,
                             backend: str = "auto") -> torch.Tensor:
    """Dense causal attention over the prompt, (1,S,Hq,D) -> (1,S,Hq,D), in place of
    flash_attn_func (reference dram_attention.py:136).  ``backend``:
      "native"  the library's kernel (16-bit types, head_dim 64 or 128; raises otherwise)
      "sdpa"    torch's fused scaled_dot_product_attention (raises if no fused kernel
                takes the shape)
      "blocked" torch's attention over blocks of query rows with an explicit mask, the
                block sized so that the scores torch may materialise for it (Hq x rows x S
                fp32) stay within 1 GiB: at most 1024 rows, 64 at 128K tokens and 32
                heads (any type, CPU too)
      "auto"    native where it applies, the library's fp32 kernel for fp32 layers with
                head_dim 64 or 128, else sdpa, else blocked."""
    if backend not in ("auto", "native", "sdpa", "blocked"):
        raise RuntimeError(f"Unsupported prefill backend: {backend}")
    if backend == "native" or (backend == "auto" and prefill_attention_supported(xq)):
        return prefill_attention(xq, xk, xv)
    if backend == "auto" and prefill_attention_f32_supported(xq, xk, xv):
        return prefill_attention_f32(xq, xk, xv)
    bsz, S, Hq, D = xq.shape
    Hkv = xk.shape[2]
    q = xq.transpose(1, 2)
    k = xk.transpose(1, 2)
    v = xv.transpose(1, 2)
    gqa = Hq != Hkv
    if backend == "sdpa" or (backend == "auto" and xq.is_cuda):
        from torch.nn.attention import SDPBackend, sdpa_kernel

        try:
            with sdpa_kernel([SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION]):
                o = F.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=gqa)
            return o.transpose(1, 2).contiguous()
        except RuntimeError:
            if backend == "sdpa":
                raise
    out = torch.empty_like(xq)
    block = max(16, min(1024, (1 << 28) // max(1, Hq * S)))
    for s0 in range(0, S, block):
        s1 = min(S, s0 + block)
        # rows s0..s1 see keys 0..s1; row i of the block may look at key j <= s0 + i
        mask = torch.ones(s1 - s0, s1, dtype=torch.bool, device=xq.device).tril_(diagonal=s0)
        o = F.scaled_dot_product_attention(q[:, :, s0:s1], k[:, :, :s1], v[:, :, :s1],
                                           attn_mask=mask, enable_gqa=gqa)
        out[:, s0:s1] = o.transpose(1, 2)
    return out


class DRAMAttention(torch.nn.Module):
    """Drop-in for the reference module of the same name.

    Two caches: ``cache_k/cache_v`` hold the local window (last
    ``local_cache_size`` prompt tokens, rounded to pages, plus everything
    generated); the rest of the prompt is paged, in host DRAM behind an
    ``LRUCache`` (or entirely in HBM behind a ``DummyCache`` when it fits
    into ``lru_hbm_cache_size``).
    """

    def __init__(
        self,
        max_output_length: int,
        lru_hbm_cache_size: int,
        local_cache_size: int,
        page_size: int,
        top_k: int,
        n_kv_heads: int,
        head_dim: int,
        device: str = "cuda",
        dtype: torch.dtype = torch.bfloat16,
    ):
        super().__init__()
        self.max_output_length = max_output_length
        self.page_size = page_size
        self.dram_kv_cache_size = None  # set by init_cache
        self.lru_hbm_cache_size = lru_hbm_cache_size
        self.local_cache_size = local_cache_size
        self.top_k = top_k
        self.n_kv_heads = n_kv_heads
        self.head_dim = head_dim
        self.num_page = self.lru_hbm_cache_size // self.page_size
        self.device = device
        cache_shape = (1, local_cache_size + max_output_length, n_kv_heads, head_dim)
        self.register_buffer("cache_k", torch.zeros(cache_shape, device=device, dtype=dtype))
        self.register_buffer("cache_v", torch.zeros(cache_shape, device=device, dtype=dtype))
        self._workspace = None
        self._side_stream = None
        # run the page stream and the first attention pass concurrently (two streams)
        self.overlap_page_stream = True
        # attend over the streamed pages inside the page stream itself (when the
        # shape allows) instead of a pass over them after the stream
        self.attend_on_page_stream = True
        # "resident": the prefix pass covers every slot of the page cache, as the
        # reference does (dram_attention.py:195-205).  "selected": only the pages this
        # step selected, each query head over its own list: the Quest baseline the
        # reference compares itself with (evaluation/quest/model.py:263-316), on the
        # same page cache and kernels.
        self.attention_scope = "resident"
        # "bound": pages ranked by the min/max upper bound (topk_selector.py:37-61 of the
        # reference).  "token_max": by the best token of each page, the accuracy ceiling
        # of page selection (evaluation/quest-top-k-oracle/model.py:267-275); keeps all
        # prefix keys on the device.  Read by init_cache.
        self.page_selector = "bound"
        # Workgroups of the page stream in all, and two rates of the machine (GB/s) that
        # time the stream + attention launch: what a kernel's reads of the pinned store
        # reach (set by init_cache from one timed pinned copy; a kernel gets about 0.95
        # of a copy engine's rate) and what one workgroup alone reads from HBM (0 = the
        # library's default).  Results do not depend on any of the three.
        self.stream_blocks = GATHER_BLOCKS
        # which implementation stage="prefill" attends with: see causal_prefill_attention
        self.prefill_backend = "auto"
        self.link_gbps = 0.0
        self.block_gbps = 0.0

    def init_cache(self, k_cache: torch.Tensor, v_cache: torch.Tensor):
        """Split the prompt's (1,S,Hkv,D) keys/values into the paged prefix and the
        local window, and build the page cache."""
        self._build_cache(k_cache, v_cache)

    def _build_cache(self, k_cache: torch.Tensor, v_cache: torch.Tensor, **build):
        """init_cache; ``build``: where an LRUCache writes its page store.  The layer changes only
        when every part is made, so a prompt that is refused leaves it as it was."""
        bsz, seqlen, H, D = k_cache.shape
        assert bsz == 1, "Only support batch size 1"
        paged = self._paged_tokens(seqlen)
        prefix_k = k_cache[0, :paged].transpose(0, 1)
        prefix_v = v_cache[0, :paged].transpose(0, 1)
        link_gbps = cache = held = None
        filled = []

        def fill(cache=None):
            # (looked at when the store and attention are on their way.  Another kind of page cache or
            # selector may still refuse the prompt behind the launch, or may not take what it makes)
            if (self.page_selector != "bound" or not self._caches_in_one_launch(k_cache, v_cache, paged)
                    or cache is not None and cache.current_step.device != k_cache.device):
                return None
            filled.append(True)
            return self._fill_caches(k_cache, v_cache, paged, cache)

        try:
            if paged > self.lru_hbm_cache_size:
                if self.page_selector not in ("bound", "token_max"):
                    raise RuntimeError(f"Unsupported page selector: {self.page_selector}")
                # (measured ahead of the store, which may be crossing the link when LRUCache returns)
                link_gbps = 0.95 * host_link_gbps(self.cache_k.device)
                if LRUCache.__init__ is _LRU_CACHE_INIT:
                    build["fill"] = fill
                cache = LRUCache(
                    k_cache=prefix_k,
                    v_cache=prefix_v,
                    page_size=self.page_size,
                    top_k=self.top_k // self.page_size,
                    lru_hbm_cache_size=self.lru_hbm_cache_size,
                    device=self.device,
                    **build,
                )
                if self.page_selector == "token_max":
                    cache.top_k_selector = TokenMaxTopKSelector(
                        prefix_k, cache.num_dram_pages, device=self.device)
            else:
                cache = DummyCache(k_cache=prefix_k, v_cache=prefix_v, device=self.device)
                fill()
            if not filled:
                tail = seqlen - paged
                window_k, window_v = self.cache_k[:, :tail], self.cache_v[:, :tail]
                tail_k, tail_v = k_cache[:, paged:], v_cache[:, paged:]
                if not tail_k.shape == tail_v.shape == window_k.shape:
                    # (both are refused here or neither is)
                    tail_k, tail_v = tail_k.expand_as(window_k), tail_v.expand_as(window_v)
                window_k.copy_(tail_k, non_blocking=True)
                window_v.copy_(tail_v, non_blocking=True)
            # Nothing refuses the prompt from here on.  The old cache is taken apart while the
            # new store is on its way, but for its own store, in pinned memory, which launches
            # of the last steps may still be reading until finish_build has waited.
            if link_gbps is not None:
                held, self.link_gbps = self._modules.get("lru_cache"), link_gbps
                held = None if held is None else held._buffers.get("dram_kv_cache")
            self.lru_cache, self.dram_kv_cache_size, self._workspace = cache, paged, None
        finally:
            if isinstance(cache, LRUCache):
                cache.finish_build()
        del held

    def _caches_in_one_launch(self, k, v, paged: int) -> bool:
        """Whether da_prompt_cache may fill this layer's window (and page cache) from a prompt's (1,S,H,D)
        keys and values: plain GPU tensors of the window's type on its device, aligned, one layout for
        both, of the size that the window was made for."""
        own = self._buffers
        cache_k, cache_v = own.get("cache_k"), own.get("cache_v")
        if cache_k is None or cache_v is None:      # (a window that is no buffer any more)
            return False
        tail, esize = k.shape[1] - paged, k.element_size()
        return (paged >= 0 and 0 <= tail <= cache_k.shape[1] and k.is_cuda and k.shape == v.shape
                and k.stride() == v.stride() and k.stride(3) == 1
                and all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.dtype is cache_k.dtype
                        and t.device == cache_k.device for t in (k, v, cache_v))
                and cache_k.shape == cache_v.shape and cache_k.shape[2:] == k.shape[2:]
                and cache_k.is_contiguous() and cache_v.is_contiguous()
                and all(n * esize % 16 == 0 for n in (k.stride(1), k.stride(2), k.shape[3]))
                and all(t.data_ptr() % 16 == 0 for t in (k, v, cache_k, cache_v))
                and not (torch.is_grad_enabled() and (k.requires_grad or v.requires_grad))
                and torch.device(self.device).type == "cuda" and unobserved())

    def _fill_caches(self, k, v, paged: int, cache=None):
        """The local window (and ``cache``'s metadata and the page summaries, returned) in one launch."""
        _, S, H, D = k.shape
        summaries, page = None, [0, None, None, None, None, None]
        if cache is not None:
            b = cache._buffers
            summaries = torch.empty(H, cache.num_dram_pages, 2, D, dtype=k.dtype, device=k.device)
            page = [cache.num_hbm_pages, summaries.data_ptr()] + [b[n].data_ptr() for n in (
                "current_step", "page_access_time", "dram_page_to_hbm_page_mapping", "hbm_page_to_dram_page_mapping")]
        _lib.check(
            _lib.load().da_prompt_cache(
                k.data_ptr(), v.data_ptr(), k.stride(1), k.stride(2), S, H, D, _lib.dtype_code(k.dtype),
                paged // self.page_size, self.page_size, *page, self._buffers["cache_k"].data_ptr(),
                self._buffers["cache_v"].data_ptr(), _lib.stream_ptr(k.device)),
            "da_prompt_cache")
        return summaries

    def _paged_tokens(self, seqlen: int) -> int:
        """Prompt tokens that go to the paged prefix; the rest is the local window."""
        return (seqlen - self.local_cache_size + self.page_size) // self.page_size * self.page_size

    def _attend_selected(self, xq, xk, xv, cache_len, offset, idx, out):
        """The Quest baseline's attention (evaluation/quest/model.py:263-316): query head
        j attends over the pages of ITS top-k list, plus the local window and the new
        token; the two partial results are combined by their log-sum-exp.  A comparison
        variant, not the hot path: the selected pages are gathered from their slots by
        torch ops and the two passes are separate calls of the decode kernel."""
        lru = self.lru_cache
        Hq, D = xq.shape[2], xq.shape[3]
        Hkv, K = idx.shape
        if K > lru.num_hbm_pages:
            raise RuntimeError("the selected-pages scope needs every selected page resident: "
                               f"{K} requests per kv head exceed {lru.num_hbm_pages} slots")
        lru.gather_(K)                                   # the missed pages land in their slots
        slots = torch.gather(lru.dram_page_to_hbm_page_mapping, 1, idx)        # (Hkv, rep*kp)
        pages = lru.hbm_kv_cache
        sel = torch.gather(pages, 1, slots[..., None].expand(-1, -1, pages.shape[2]))
        sel = sel.view(Hq, (K // (Hq // Hkv)) * self.page_size, 2, D)   # rows of q head h*rep + r
        no_cache = xq.new_empty(0, Hq, D)
        lse_p = torch.empty(Hq, dtype=torch.float32, device=xq.device)
        lse_s = torch.empty_like(lse_p)
        out_p = decode_attention(xq[0, 0], sel[:, :, 0], sel[:, :, 1], no_cache, no_cache, 0, None,
                                 None, lse=lse_p)
        out_s = decode_attention(xq[0, 0], None, None, self.cache_k[0], self.cache_v[0], cache_len,
                                 xk[0, 0], xv[0, 0], lse=lse_s, cache_len_offset=offset)
        lse = torch.logaddexp(lse_p, lse_s)
        mixed = (out_p.float() * torch.exp(lse_p - lse)[:, None]
                 + out_s.float() * torch.exp(lse_s - lse)[:, None])
        out[0, 0].copy_(mixed)

    def init_cache_from_file(self, cache_dir: str, index: int) -> int:
        """init_cache from the chat example's per-layer file ``NN_cache.pth``; returns
        the prompt length (the position of the first generated token)."""
        from .kv_file import load_layer_cache

        k, v = load_layer_cache(cache_dir, index, self.device)
        self.init_cache(k.to(self.cache_k.dtype), v.to(self.cache_v.dtype))
        return k.shape[1]

    def forward(self, xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor, *, start_pos,
                stage: str):
        bsz, seqlen, H, D = xq.shape
        assert bsz == 1, "Only support batch size 1"
        if stage == "prefill":
            return self._prefill(xq, xk, xv)
        elif stage == "generate":
            return self._generate(xq, xk, xv, start_pos)
        else:
            raise RuntimeError(f"Unsupported stage: {stage}")

    def _prefill(self, xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor):
        """Attention over the prompt and the caches built from it.  Where a library kernel
        attends, the page store is written next to it, on a stream of its own: attention is
        bound by the matrix cores, the store by the host link.  An init_cache of somebody's
        own is called, behind attention."""
        paged = self._paged_tokens(xk.shape[1])
        if not (paged > self.lru_hbm_cache_size
                and type(self).init_cache is _INIT_CACHE and "init_cache" not in self.__dict__
                and self.prefill_backend in ("auto", "native") and xk.is_cuda
                and (prefill_attention_supported(xq) or prefill_attention_f32_supported(xq, xk, xv))):
            output = causal_prefill_attention(xq, xk, xv, self.prefill_backend)
            self.init_cache(xk, xv)
            return output
        output = []
        self._build_cache(
            xk, xv, build_stream=build_stream(xk.device),
            build_blocks=store_build_blocks(xq.shape, (1, paged, *xk.shape[2:]), xq.dtype, self.page_size,
                                            self.lru_hbm_cache_size / paged),
            beside=lambda: output.append(causal_prefill_attention(xq, xk, xv, self.prefill_backend)))
        return output[0]

    def _generate(self, xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor, start_pos):
        """One decode step: select pages, update the LRU, then one attention pass
        over resident pages, local window and the new token (appended in place).
        The missed pages stream in on a side stream while attention already
        covers the local window and every slot that keeps its page."""
        out = self._step_in_one_call(xq, xk, xv, start_pos)
        if out is not None:
            return out
        return self.attend_(xq, xk, xv, start_pos, self.select_(xq))

    def _step_in_one_call(self, xq, xk, xv, start_pos):
        """select_ and attend_ as one native call (da_decode_step; over a static prefix
        da_decode_attention) where everything has the layout a layer is built with; None where
        anything differs, and the two methods, which take or refuse it, do the step.  The same
        results on the same operands."""
        lru = self._modules.get("lru_cache")
        if type(lru) is DummyCache:
            return self._static_step(lru, xq, xk, xv, start_pos)
        step = self._step_args(xq, xk, xv, start_pos)
        if step is None:
            return None
        args, out = step
        _lib.check(_lib.load().da_decode_step(args, len(args), _lib.stream_ptr(xq.device)), "da_decode_step")
        return out

    def _static_step(self, lru, xq, xk, xv, start_pos):
        """A step over a static prefix, or None (a prompt's first, too, by which the workspace is sized)."""
        if self._workspace is None:
            return None
        cls, layer, own, prefix = type(self), self.__dict__, self._buffers, lru.__dict__
        if ((cls.select_, cls.attend_, DummyCache.get_kv_cache_) != _STATIC_METHODS or "select_" in layer
                or "attend_" in layer or "get_kv_cache_" in prefix):
            return None
        return _lib.host().static_step(
            xq, xk, xv, start_pos, prefix.get("k_cache"), prefix.get("v_cache"), own.get("cache_k"),
            own.get("cache_v"), self.dram_kv_cache_size, self._workspace, _lib.stream_ptr(xq.device))

    def _step_args(self, xq, xk, xv, start_pos):
        """(argument block of da_decode_step, output) of a step that one native call can do, else None."""
        lru = self.lru_cache
        if (type(lru) is not LRUCache or self.attention_scope != "resident" or not self.overlap_page_stream
                or not self.attend_on_page_stream):
            return None
        selector, buffers, own = lru.top_k_selector, lru._buffers, self._buffers
        if type(selector) is not IPUpperboundTopKSelector or not self._steps_by_its_own_methods(lru, selector):
            return None
        step_args = _lib.host().step_args
        if not isinstance(start_pos, torch.Tensor):
            start_pos = int(start_pos)
        for _ in range(2):
            step = step_args(
                xq, xk, xv, start_pos, selector.chunk_min_max, buffers["dram_kv_cache"], buffers["hbm_kv_cache"],
                buffers["page_access_time"], buffers["dram_page_to_hbm_page_mapping"],
                buffers["hbm_page_to_dram_page_mapping"], buffers["current_step"], own.get("cache_k"),
                own.get("cache_v"), lru.num_hbm_pages, lru.page_size, lru.top_k, self.dram_kv_cache_size, lru.page_stores()[1],
                self.stream_blocks, SCORE_FLAGS[selector.bounds_are_ordered], self.link_gbps, self.block_gbps,
                lru._scratch, lru._topk_idx, selector._scores, selector._split_ws, self._workspace)
            if type(step) is not int:
                return step
            self._make_room(lru, selector, step, xq)    # (a layer's first step)
        return None

    def _make_room(self, lru, selector, rep, xq):
        """What the launches of a step hand to one another, for ``rep`` query rows a kv head."""
        H, P, _, D = selector.chunk_min_max.shape
        kp, device = min(lru.top_k, P), xq.device

        def room(t, shape, dtype):
            if t is not None and t.shape == shape and t.dtype is dtype and t.device == device and t.is_contiguous():
                return t
            return torch.empty(shape, dtype=dtype, device=device)

        lru._scratch_for(rep * kp)
        lru._topk_idx = room(lru._topk_idx, (H, rep * kp), torch.int64)
        selector._scores = room(selector._scores, (rep, H, P), torch.float32)
        selector._workspace(selector._scores, kp)
        if self._workspace is None:
            self._workspace = attention_workspace(
                rep * H, H, D, xq.dtype, lru.num_hbm_pages * lru.page_size, self.cache_k.shape[1],
                rep * kp * lru.page_size, device)

    def _steps_by_its_own_methods(self, lru, selector) -> bool:
        """Whether the methods a step is made of are this module's: neither a subclass, nor an
        exchanged method of a class, the layer, its page cache or its selector would be passed by."""
        cls, layer, cache, ranking = type(self), self.__dict__, lru.__dict__, selector.__dict__
        return ((cls.select_, cls.attend_, LRUCache.select_, LRUCache.update_, LRUCache.views,
                 IPUpperboundTopKSelector.top_k_for_lru, IPUpperboundTopKSelector.scores) == _STEP_METHODS
                and not ("select_" in layer or "attend_" in layer or "select_" in cache or "update_" in cache
                         or "views" in cache or "top_k_for_lru" in ranking or "scores" in ranking))

    def select_(self, xq: torch.Tensor):
        """First half of a decode step: page scores, ordered top-k and the LRU update
        (three launches that touch neither the host link nor K/V).  Returns what
        :meth:`attend_` needs to finish the step, or None with a static cache.  The
        two halves may be issued on different streams as long as attend_ is ordered
        after select_ of the same step and before select_ of the next one."""
        bsz, seqlen, Hq, D = xq.shape
        if seqlen != 1:
            raise RuntimeError("generate handles one token per call")
        lru = self.lru_cache
        if not isinstance(lru, LRUCache):
            return None
        idx = lru.select_(xq)
        return idx, lru.update_(idx)

    def attend_(self, xq: torch.Tensor, xk: torch.Tensor, xv: torch.Tensor, start_pos, selected,
                defer_merge: bool = False):
        """Second half of a decode step: the page stream for the misses select_ found
        and attention over resident pages, local window and the new token.
        ``defer_merge``: when the step's final merge is a launch of its own (page
        stream and first pass in one launch), leave it out and return (out, merge)
        where ``merge()`` issues it on whatever stream is current, ordered after
        this call; ``out`` is complete only then.  Otherwise returns (out, None)."""
        bsz, seqlen, Hq, D = xq.shape
        if seqlen != 1:
            raise RuntimeError("generate handles one token per call")
        if isinstance(start_pos, torch.Tensor):
            # the position stays on the device; the kernel subtracts the paged prefix
            cache_len = start_pos if start_pos.dtype == torch.int32 else start_pos.to(torch.int32)
            offset = -self.dram_kv_cache_size
        else:
            cache_len, offset = int(start_pos) - self.dram_kv_cache_size, 0
        out = torch.empty(1, 1, Hq, D, dtype=xq.dtype, device=xq.device)
        lru = self.lru_cache
        if not isinstance(lru, LRUCache):
            prefix_k, prefix_v = lru.get_kv_cache_(xq)
            if self._workspace is None:
                self._workspace = attention_workspace(Hq, self.n_kv_heads, D, xq.dtype,
                                                      prefix_k.shape[1], self.cache_k.shape[1], 0,
                                                      xq.device)
            decode_attention(xq[0, 0], prefix_k, prefix_v, self.cache_k[0], self.cache_v[0],
                             cache_len, xk[0, 0], xv[0, 0], workspace=self._workspace,
                             out=out[0, 0], cache_len_offset=offset)
            return (out, None) if defer_merge else out

        idx, scratch = selected
        if self.attention_scope == "selected":
            self._attend_selected(xq, xk, xv, cache_len, offset, idx, out)
            return (out, None) if defer_merge else out
        if self.attention_scope != "resident":
            raise RuntimeError(f"Unsupported attention scope: {self.attention_scope}")
        prefix_k, prefix_v = lru.views()
        if self._workspace is None:
            self._workspace = attention_workspace(
                Hq, self.n_kv_heads, D, xq.dtype, prefix_k.shape[1], self.cache_k.shape[1],
                scratch.miss_slot.shape[1] * self.page_size, xq.device)
        args = (xq[0, 0], prefix_k, prefix_v, self.cache_k[0], self.cache_v[0], cache_len,
                xk[0, 0], xv[0, 0])
        k = idx.shape[1]
        # Attention over the pages paged in this step rides on the page stream when
        # the shape allows; otherwise a tail pass covers them after the stream.
        fused = self.attend_on_page_stream and gather_attend_supported(
            Hq, self.n_kv_heads, D, self.page_size, xq.dtype)
        blocks = max(1, min(self.stream_blocks // self.n_kv_heads, k)) if fused else 0

        def stream_pages():
            if fused:
                lru.gather_attend_(k, xq[0, 0], 1.0 / math.sqrt(D), self.cache_k.shape[1],
                                   self._workspace, blocks)
            else:
                lru.gather_(k)

        def attend(phase):
            decode_attention(*args, workspace=self._workspace, out=out[0, 0],
                             cache_len_offset=offset,
                             paged=PagedPrefix(self.page_size, scratch, lru.current_step, phase,
                                               blocks))

        P = PagedPrefix
        if not self.overlap_page_stream:
            stream_pages()
            # the same kernels as the concurrent order, so the same bits
            attend((P.FIRST | P.SECOND) if fused else (P.FIRST | P.FIRST_MERGE | P.SECOND))
            return (out, None) if defer_merge else out
        if fused:
            # page stream and first attention pass in one launch, then the merge: the
            # step stays a plain chain of launches on the caller's stream
            def launch(phase):
                decode_attention(*args, workspace=self._workspace, out=out[0, 0],
                                 cache_len_offset=offset,
                                 paged=PagedPrefix(self.page_size, scratch, lru.current_step,
                                                   phase, blocks, lru.page_stores(),
                                                   self.link_gbps, self.block_gbps))

            if defer_merge:
                launch(P.STREAM | P.FIRST)
                return out, (lambda: launch(P.SECOND | P.MERGE_ALL))
            launch(P.STREAM | P.FIRST | P.SECOND)
            return out
        # Shapes the fused stream does not take: pages stream in on a side stream
        # next to the first pass, and a tail pass covers them after the join.
        main = torch.cuda.current_stream(xq.device)
        if self._side_stream is None:
            self._side_stream = torch.cuda.Stream(device=xq.device)
        side = self._side_stream
        side.wait_stream(main)                      # the miss list is ready
        with torch.cuda.stream(side):
            stream_pages()
        attend(P.FIRST | P.FIRST_MERGE)
        main.wait_stream(side)                      # the pages have landed
        attend(P.SECOND)
        return (out, None) if defer_merge else out


_STEP_METHODS = (DRAMAttention.select_, DRAMAttention.attend_, LRUCache.select_, LRUCache.update_, LRUCache.views,
                 IPUpperboundTopKSelector.top_k_for_lru, IPUpperboundTopKSelector.scores)
_STATIC_METHODS = (DRAMAttention.select_, DRAMAttention.attend_, DummyCache.get_kv_cache_)
_INIT_CACHE = DRAMAttention.init_cache
_LRU_CACHE_INIT = LRUCache.__init__
