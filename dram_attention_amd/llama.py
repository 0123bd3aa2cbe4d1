"""Llama-3 shaped decoder whose attention layers are ``DRAMAttention``.

Counterpart of the model the reference evaluates with
(evaluation/dram-attention/model.py:28-317): same ``ModelArgs`` fields, same
module and parameter names (``tok_embeddings``, ``layers.N.attention.wq`` …
``norm``, ``output``), so a Llama-3 checkpoint's state dict loads unchanged,
and the same ``forward(tokens, start_pos)`` contract: a call with more than one
token at position 0 is the prefill (it builds every layer's page cache), any
other call decodes one token.  ``start_pos`` of a decode call may be an int32
device tensor, which keeps the step free of host reads so that it can be
captured in a HIP graph the way examples/long-qa-chat/chat.py:238-249 does.

Projections of a prompt are torch's linear layers; norms, rotary embedding and
SwiGLU, and the whole block around the attention of a single token, run in the
kernels of ``model_kernels`` where those take the tensors, and in torch's operators
otherwise (the CPU, autograd, hooked or replaced modules), with the same roundings.
"""
from __future__ import annotations

import math
from dataclasses import dataclass
from typing import Optional

import torch
import torch.nn.functional as F
from torch import nn

from . import model_kernels as K
from .dram_attention import DRAMAttention


@dataclass
class ModelArgs:
    """Model and cache geometry; defaults are Llama-3.1-8B with the reference's
    cache settings (evaluation/dram-attention/model.py:28-63)."""

    dim: int = 4096
    n_layers: int = 32
    n_heads: int = 32
    n_kv_heads: Optional[int] = None
    vocab_size: int = -1
    multiple_of: int = 256
    ffn_dim_multiplier: Optional[float] = None
    norm_eps: float = 1e-5
    rope_theta: float = 500000
    use_scaled_rope: bool = False
    lru_hbm_cache_size: int = 32 * 1024
    local_cache_size: int = 4 * 1024 + 1024
    cache_page_size: int = 16
    cache_top_k: int = 4 * 1024
    max_output_length: int = 128
    max_batch_size: int = 1
    max_seq_len: int = 2048
    dtype: torch.dtype = torch.bfloat16
    # which of the reference's evaluated models the attention layers form:
    #   "dram"  DRAM Attention (evaluation/dram-attention/model.py)
    #   "quest" attention over the selected pages only (evaluation/quest/model.py:263-316)
    #   "quest_oracle" the same with pages ranked by their best token instead of the
    #           min/max bound (evaluation/quest-top-k-oracle/model.py:267-275)
    #   "full"  dense attention over the whole cache (evaluation/full-attention/model.py:201-215)
    attention_variant: str = "dram"

    def __post_init__(self):
        if self.n_kv_heads is None:
            self.n_kv_heads = self.n_heads
        assert self.n_kv_heads <= self.n_heads
        assert self.n_heads % self.n_kv_heads == 0
        assert self.dim % self.n_heads == 0
        assert self.attention_variant in ("dram", "quest", "quest_oracle", "full")

    @property
    def head_dim(self) -> int:
        return self.dim // self.n_heads


def ffn_hidden_dim(dim: int, multiple_of: int, ffn_dim_multiplier: Optional[float]) -> int:
    """Width of the SwiGLU layer: 2/3 of 4*dim, scaled, rounded up to ``multiple_of``
    (evaluation/dram-attention/model.py:216-220)."""
    hidden = int(2 * (4 * dim) / 3)
    if ffn_dim_multiplier is not None:
        hidden = int(ffn_dim_multiplier * hidden)
    return multiple_of * ((hidden + multiple_of - 1) // multiple_of)


def rope_frequencies(head_dim: int, theta: float, use_scaled: bool) -> torch.Tensor:
    """The head_dim/2 rotation frequencies; with ``use_scaled`` the Llama-3.1
    long-context rule: wavelengths above 8192 slowed 8x, below 2048 kept, a linear
    blend between (evaluation/dram-attention/model.py:81-105)."""
    freqs = 1.0 / (theta ** (torch.arange(0, head_dim, 2)[: head_dim // 2].float() / head_dim))
    if not use_scaled:
        return freqs
    scale, low, high, old_len = 8.0, 1.0, 4.0, 8192.0
    wavelen = 2 * math.pi / freqs
    smooth = ((old_len / wavelen - low) / (high - low)).clamp(0.0, 1.0)
    # smooth is 0 for wavelengths above old_len/low and 1 below old_len/high
    return (1 - smooth) * freqs / scale + smooth * freqs


def rope_table(head_dim: int, end: int, theta: float, use_scaled: bool,
               device=None) -> torch.Tensor:
    """(end, head_dim/2, 2) fp32: cos and sin of position * frequency."""
    angle = torch.outer(torch.arange(end, dtype=torch.float32),
                        rope_frequencies(head_dim, theta, use_scaled))
    return torch.stack((angle.cos(), angle.sin()), dim=-1).to(device)


def apply_rope(x: torch.Tensor, rows: torch.Tensor) -> torch.Tensor:
    """Rotate adjacent channel pairs of x (1, S, H, D) by the table rows (S, D/2, 2);
    arithmetic in fp32, result in x's dtype (the complex product of
    evaluation/dram-attention/model.py:126-136 written out)."""
    pairs = x.float().unflatten(-1, (-1, 2))
    even, odd = pairs[..., 0], pairs[..., 1]
    cos, sin = rows[None, :, None, :, 0], rows[None, :, None, :, 1]
    out = torch.stack((even * cos - odd * sin, even * sin + odd * cos), dim=-1)
    return out.flatten(-2).to(x.dtype)


class RMSNorm(nn.Module):
    def __init__(self, dim: int, eps: float = 1e-6):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim))

    def forward(self, x):
        if K.takes(x, self.weight) and K.norm_fits(x, self.weight):
            return K.rms_norm(x, self.weight, self.eps)[0]
        x32 = x.float()
        normed = x32 * torch.rsqrt(x32.square().mean(-1, keepdim=True) + self.eps)
        return normed.to(x.dtype) * self.weight

    def after_add(self, x, y):
        """(norm of x + y, x + y)."""
        if K.takes(x, y, self.weight) and K.norm_fits(x, self.weight) and x.shape == y.shape:
            return K.rms_norm(x, self.weight, self.eps, add=y)
        total = x + y
        return self(total), total


class Attention(nn.Module):
    """Projections and rotary embedding around DRAMAttention
    (evaluation/dram-attention/model.py:138-205)."""

    def __init__(self, args: ModelArgs, device="cuda"):
        super().__init__()
        self.n_heads, self.n_kv_heads, self.head_dim = args.n_heads, args.n_kv_heads, args.head_dim
        self.wq = nn.Linear(args.dim, args.n_heads * self.head_dim, bias=False)
        self.wk = nn.Linear(args.dim, args.n_kv_heads * self.head_dim, bias=False)
        self.wv = nn.Linear(args.dim, args.n_kv_heads * self.head_dim, bias=False)
        self.wo = nn.Linear(args.n_heads * self.head_dim, args.dim, bias=False)
        # "full": a page cache as large as the longest sequence keeps the whole prefix
        # in HBM (init_cache then picks the static cache: plain dense attention)
        budget = (max(args.lru_hbm_cache_size, args.max_seq_len)
                  if args.attention_variant == "full" else args.lru_hbm_cache_size)
        self.dram_attention = DRAMAttention(
            max_output_length=args.max_output_length,
            lru_hbm_cache_size=budget,
            local_cache_size=args.local_cache_size,
            page_size=args.cache_page_size,
            top_k=args.cache_top_k,
            n_kv_heads=args.n_kv_heads,
            head_dim=self.head_dim,
            device=device,
            dtype=args.dtype,
        )
        if args.attention_variant in ("quest", "quest_oracle"):
            self.dram_attention.attention_scope = "selected"
        if args.attention_variant == "quest_oracle":
            self.dram_attention.page_selector = "token_max"

    def forward(self, x: torch.Tensor, start_pos, rope_rows: torch.Tensor):
        bsz, seqlen, _ = x.shape
        xq = self.wq(x).view(bsz, seqlen, self.n_heads, self.head_dim)
        xk = self.wk(x).view(bsz, seqlen, self.n_kv_heads, self.head_dim)
        xv = self.wv(x).view(bsz, seqlen, self.n_kv_heads, self.head_dim)
        if (K.takes(xq, xk) and K.plain_linears(self.wq, self.wk) and rope_rows.dtype == torch.float32
                and rope_rows.is_contiguous() and rope_rows.device == xq.device and rope_rows.data_ptr() % 16 == 0
                and bsz == 1 and rope_rows.shape == (seqlen, self.head_dim // 2, 2)
                and self.head_dim * xq.element_size() % 16 == 0):
            K.rope_(xq, xk, rope_rows)          # the projections' own outputs, in place
        else:
            xq, xk = apply_rope(xq, rope_rows), apply_rope(xk, rope_rows)
        prefill = seqlen > 1 and not isinstance(start_pos, torch.Tensor) and start_pos == 0
        out = self.dram_attention(xq, xk, xv, start_pos=start_pos,
                                  stage="prefill" if prefill else "generate")
        return self.wo(out.reshape(bsz, seqlen, -1))


class FeedForward(nn.Module):
    ROWS_PER_PASS = 8192  # a long prompt goes through in slices (model.py:236-245)

    def __init__(self, dim: int, multiple_of: int, ffn_dim_multiplier: Optional[float]):
        super().__init__()
        hidden = ffn_hidden_dim(dim, multiple_of, ffn_dim_multiplier)
        self.w1 = nn.Linear(dim, hidden, bias=False)
        self.w2 = nn.Linear(hidden, dim, bias=False)
        self.w3 = nn.Linear(dim, hidden, bias=False)

    def forward(self, x):
        if x.shape[1] <= self.ROWS_PER_PASS:
            return self._slice(x)
        return torch.cat([self._slice(c) for c in x.split(self.ROWS_PER_PASS, dim=1)], dim=1)

    def _slice(self, x):
        gate, up = self.w1(x), self.w3(x)
        if (K.takes(gate, up) and K.plain_linears(self.w1) and gate.shape == up.shape
                and gate.numel() * gate.element_size() % 16 == 0):
            return self.w2(K.swiglu_(gate, up))     # in w1's own output
        return self.w2(F.silu(gate) * up)


class TransformerBlock(nn.Module):
    def __init__(self, layer_id: int, args: ModelArgs, device="cuda"):
        super().__init__()
        self.layer_id = layer_id
        self.attention = Attention(args, device)
        self.feed_forward = FeedForward(args.dim, args.multiple_of, args.ffn_dim_multiplier)
        self.attention_norm = RMSNorm(args.dim, eps=args.norm_eps)
        self.ffn_norm = RMSNorm(args.dim, eps=args.norm_eps)

    def forward(self, x, start_pos, rope_rows):
        if x.shape[0] == x.shape[1] == 1:
            parts = self._modules
            a, f, norm1, norm2 = (parts["attention"], parts["feed_forward"], parts["attention_norm"],
                                  parts["ffn_norm"])
            weights = self._one_token_kernels(a, f, norm1, norm2, x, rope_rows)
            if weights is not None:
                wq, wk, wv, wo, w1, w3, w2 = weights
                xq, xk, xv = K.linear_qkv_rope(x, norm1, wq, wk, wv, a.n_heads, a.n_kv_heads, a.head_dim,
                                               rope_rows)
                out = a.dram_attention(xq, xk, xv, start_pos=start_pos, stage="generate")
                if K.row_fits(out, x, wo.shape[1]):
                    return K.block_tail(out, wo, x, norm2, w1, w3, w2)
                # (an attention module of its own kind, or a hook, returned something else)
                return self._tail(x, a.wo(out.reshape(1, 1, -1)))
        return self._tail(x, self.attention(self.attention_norm(x), start_pos, rope_rows))

    def _tail(self, x, attended):
        """Residuals and feed-forward behind attention's projected output."""
        if type(self.ffn_norm) is RMSNorm and K.bare(self.ffn_norm):
            normed, h = self.ffn_norm.after_add(x, attended)
        else:
            h = x + attended
            normed = self.ffn_norm(h)
        return h + self.feed_forward(normed)

    @staticmethod
    def _one_token_kernels(a, f, norm1, norm2, x, rope_rows):
        """The weights (wq, wk, wv, wo, w1, w3, w2) if the one-token kernels may stand for these
        modules of a block, else None: the modules are the block's own kinds, nobody watches
        them, and every shape is the one that the kernels take for granted."""
        if not (type(a) is Attention and type(f) is FeedForward and type(norm1) is type(norm2) is RMSNorm):
            return None
        weight1, weight2 = norm1._parameters.get("weight"), norm2._parameters.get("weight")
        if not (K.takes(x, weight1, weight2) and K.bare(a, f, norm1, norm2)
                and type(rope_rows) in (torch.Tensor, nn.Parameter) and rope_rows.dtype is torch.float32 and rope_rows.is_contiguous()
                and rope_rows.device == x.device):
            return None
        am, fm, dim, hd = a._modules, f._modules, x.shape[2], a.head_dim
        w1 = fm["w1"]
        q_rows, kv_rows, hidden = a.n_heads * hd, a.n_kv_heads * hd, getattr(w1, "out_features", -1)
        if not (dim * x.element_size() % 16 == 0 and weight1.shape == weight2.shape == (dim,)
                and rope_rows.shape == (1, hd // 2, 2) and hd % 2 == 0):
            return None
        return K.linears_fit(x, (am["wq"], q_rows, dim), (am["wk"], kv_rows, dim), (am["wv"], kv_rows, dim),
                             (am["wo"], dim, q_rows), (w1, hidden, dim), (fm["w3"], hidden, dim),
                             (fm["w2"], dim, hidden))


def _index(position: torch.Tensor) -> torch.Tensor:
    """A device position as one index (32 bits are one as they are: no launch)."""
    index = position.reshape(1)
    return index if index.dtype in (torch.int32, torch.int64) else index.long()


class Transformer(nn.Module):
    """``forward(tokens (1, S), start_pos) -> logits (1, 1, vocab)`` fp32 of the last
    position (evaluation/dram-attention/model.py:276-317)."""

    def __init__(self, params: ModelArgs, device="cuda"):
        super().__init__()
        self.params = params
        with torch.device(device):  # parameters are born on the device
            self.tok_embeddings = nn.Embedding(params.vocab_size, params.dim)
            self.layers = nn.ModuleList(TransformerBlock(i, params, device)
                                        for i in range(params.n_layers))
            self.norm = RMSNorm(params.dim, eps=params.norm_eps)
            self.output = nn.Linear(params.dim, params.vocab_size, bias=False)
        with torch.device("cpu"):   # one table for every device: built on the host
            rope = rope_table(params.head_dim, params.max_seq_len * 2, params.rope_theta,
                              params.use_scaled_rope)
        self.rope = rope.to(device)
        self.to(dtype=params.dtype)

    @torch.no_grad()
    def forward(self, tokens: torch.Tensor, start_pos):
        _bsz, seqlen = tokens.shape
        h = self.tok_embeddings(tokens)
        if isinstance(start_pos, torch.Tensor):
            assert seqlen == 1, "a device-resident position is for single-token decode steps"
            rows = self.rope.index_select(0, _index(start_pos))
        else:
            rows = self.rope[start_pos: start_pos + seqlen]
        for layer in self.layers:
            h = layer(h, start_pos, rows)
        last = h[:, -1:, :]
        if (last.shape[0] == 1 and K.takes(last, self.norm.weight) and K.linears_fit(last, self.output)
                and type(self.norm) is RMSNorm and K.bare(self.norm)
                and self.output.in_features == last.shape[2] and self.norm.weight.shape == last.shape[2:]):
            return K.linear_logits(last, self.norm, self.output.weight)
        return self.output(self.norm(last)).float()

    def init_cache_from_files(self, cache_dir: str) -> int:
        """Load every layer's ``NN_cache.pth`` (examples/long-qa-chat/chat.py:214-233);
        returns the prompt length."""
        n = 0
        for i, layer in enumerate(self.layers):
            n = layer.attention.dram_attention.init_cache_from_file(cache_dir, i)
        return n


class GraphedDecoder:
    """Greedy decoding with the whole model step in one HIP graph, position and
    token resident on the device (examples/long-qa-chat/chat.py:238-273).

    The first step after the prompt runs eagerly: it sizes every layer's
    workspace, which a capture must not do.
    """

    def __init__(self, model: Transformer, prompt_len: int, first_token: int):
        dev = model.tok_embeddings.weight.device
        self.model = model
        self.token = torch.tensor([[first_token]], dtype=torch.long, device=dev)
        self.pos = torch.tensor([prompt_len], dtype=torch.int32, device=dev)
        self.graph = None
        self.logits = None

    @torch.no_grad()        # (the caller's mode would otherwise keep the arg-max from its kernel)
    def _step(self):
        logits = self.model(self.token, self.pos)
        if (K.takes(logits) and logits.dtype == torch.float32 and logits.numel() == logits.shape[-1]
                and K.is_token(self.token, logits)):
            K.argmax_into(logits, self.token)
        else:
            self.token.copy_(logits.argmax(-1))
        self.pos.add_(1)
        return logits

    def step(self) -> torch.Tensor:
        """Feed the current token, advance; returns the logits (1, 1, vocab), valid
        until the next call."""
        if self.graph is None and self.logits is None:
            self.logits = self._step()
            return self.logits
        if self.graph is None:
            torch.cuda.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                self.logits = self._step()
        self.graph.replay()
        return self.logits
