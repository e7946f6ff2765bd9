"""Llama-style decoder with the SOCKET attention hook on the HIP decode path.

Host-side mirror of GPT-FAST/model.py (ModelArgs :103-136, KVCache :157-229,
Transformer :232-329, TransformerBlock :332-349, Attention :352-589,
FeedForward :592-600, RMSNorm :603-614, rotary helpers :617-639): same class,
method and argument names, same math for projections, rotary embedding, norms
and the soft / hard hashes.  What differs is how the attention hook keeps and
walks its state:

  * the cache stores packed, table-major bucket codes per KV head
    (`KVCache.codes`, int32 [B,Hkv,NW,Tcap]) instead of int16 `k_hard`
    [B,Hkv,T,L]; new keys are hashed and their value norms taken by one kernel
    as they are appended (model.py:449-451 + :222-226 in one launch);
  * lengths live on the device (`KVCache.lens`), so a decode step reads nothing
    back to the host (the reference syncs at model.py:211-212,228,483) and the
    whole step can be recorded into a HIP graph;
  * no per-step code relayout (model.py:490-509), no K/V prefix copies
    (:541-542), no T x T boolean mask (:279-281): a 16-bit prompt attends causally
    through the HIP kernel of csrc/prompt_attend.hip (other types and head widths, and
    anything that is differentiated, through torch's SDPA), decode through the HIP kernels.

Everything outside the attention hook (embedding, linears, norms, rotary) is
plain torch: it is plumbing around the path, not part of it.
"""
from __future__ import annotations

import math
from dataclasses import dataclass
from typing import Optional, Sequence, Tuple

import torch
import torch.nn as nn
from torch import Tensor
from torch.nn import functional as F

from . import decode_ops, hash_cache, layer_ops
from .socket_kernels import dense_decode_fwd


def find_multiple(n: int, k: int) -> int:
    return n if n % k == 0 else n + k - (n % k)


@dataclass
class ModelArgs:
    """Same fields and defaults as GPT-FAST/model.py:103-118; `sink_size` and
    `window_size` are the attributes the reference reads with
    getattr(config, ..., 120) at model.py:511-512."""
    block_size: int = 300000
    vocab_size: int = 32000
    n_layer: int = 1
    n_head: int = 32
    dim: int = 4096
    intermediate_size: int = None
    n_local_heads: int = -1
    head_dim: int = 64
    rope_base: float = 40000
    norm_eps: float = 1e-5
    L: int = 60
    R: int = 1024
    K: int = 10
    heavy_const: int = 3600
    sink_size: int = 120
    window_size: int = 120
    # Not in the reference: with True a sparse decode step takes the dense kernel while
    # the cache is short enough for `hash_cache.step_cost_estimate` to price dense
    # attention below score + select + attend (exact attention, and faster there);
    # False keeps `decode_type="sparse"` sparse at every length, as the reference does.
    dense_below_crossover: bool = False

    def __post_init__(self):
        if self.n_local_heads == -1:
            self.n_local_heads = self.n_head
        if self.intermediate_size is None:
            self.intermediate_size = find_multiple(int(2 * (4 * self.dim) / 3), 256)
        self.head_dim = self.dim // self.n_head

    @classmethod
    def from_name(cls, name: str):
        if name in transformer_configs:
            return cls(**transformer_configs[name])
        hits = [c for c in transformer_configs if c in str(name).upper() or c in str(name)]
        assert len(hits) == 1, name
        return cls(**transformer_configs[hits[0]])


transformer_configs = {
    # the reference's table (GPT-FAST/model.py:138-154)
    "CodeLlama-7b-Python-hf": dict(block_size=16384, vocab_size=32000, n_layer=1, dim=4096, rope_base=1000000),
    "Llama-2-7b-chat-hf": dict(block_size=300000, vocab_size=32000, n_layer=1, n_head=32, dim=4096, rope_base=10000),
    "7B": dict(n_layer=1, n_head=32, dim=4096),
    "13B": dict(n_layer=1, n_head=40, dim=5120),
    "30B": dict(n_layer=1, n_head=52, dim=6656),
    "34B": dict(n_layer=1, n_head=64, dim=8192, vocab_size=32000, n_local_heads=8, intermediate_size=22016,
                rope_base=1000000),
    "70B": dict(n_layer=1, n_head=64, dim=8192, n_local_heads=8, intermediate_size=28672),
    # the long-context decode benchmark's model: Llama-3.1-8B geometry, random weights
    "Llama-3.1-8B": dict(block_size=131072, vocab_size=128256, n_layer=32, n_head=32, n_local_heads=8, dim=4096,
                         intermediate_size=14336, rope_base=500000, heavy_const=2048, sink_size=4,
                         window_size=256),
}


class KVCache(nn.Module):
    """K/V [B,Hkv,Tcap,D] plus the hash state of every cached key.

    Constructor as GPT-FAST/model.py:162-171 with two keyword additions (`K`,
    the bits per table, which fixes the packing; `device`).  `update` keeps the
    reference's signature and bounds error (model.py:187-229) and takes any index
    tensor; one ascending run (arange(T) for prefill, [pos] for a decode step: all
    the reference's own call path produces) is written in one piece, anything else
    as the runs it consists of.  The cached length `lens` follows the last write
    (largest position + 1) where the reference keeps a running maximum."""

    def __init__(self, max_batch_size: int, max_seq_length: int, n_heads: int, head_dim: int, L: int, R: int,
                 dtype=torch.bfloat16, K: int = 10, device=None):
        super().__init__()
        B, H, D = max_batch_size, n_heads, head_dim
        T = find_multiple(max_seq_length, 8)
        self.L, self.R, self.K = L, R, K
        self.NW = hash_cache.words_per_key(L, K)
        self.register_buffer("k_cache", torch.zeros((B, H, T, D), dtype=dtype, device=device))
        self.register_buffer("v_cache", torch.zeros((B, H, T, D), dtype=dtype, device=device))
        self.register_buffer("codes", torch.zeros((B, H, self.NW, T), dtype=torch.int32, device=device))
        self.register_buffer("v_norm", torch.zeros((B, H, T), dtype=torch.float16, device=device))
        self.register_buffer("attn_out", torch.zeros((B, H, D), dtype=dtype, device=device))
        self.register_buffer("lens", torch.zeros((B,), dtype=torch.int32, device=device))
        self.planes_words: Optional[Tensor] = None   # set by Attention once the planes are known

    @property
    def prefill_len(self) -> Tensor:
        """0-d int32 count of cached positions (the reference's buffer of that name)."""
        return self.lens.max()

    def k_hard(self, T: int) -> Tensor:
        """int16 codes [B,Hkv,T,L] as the reference's `k_hard` buffer holds them."""
        return hash_cache.unpack_codes(self.codes, self.L, self.K, 0, T, layout="bhlt").permute(0, 1, 3, 2)

    def _bounds(self, pos0: int, S: int) -> None:
        Tcap = self.k_cache.size(2)
        if pos0 < 0 or pos0 + S > Tcap:
            raise RuntimeError(
                f"KVCache.update out-of-bounds: input_pos in [{pos0},{pos0 + S - 1}] but cache T={Tcap}. "
                f"Did you call setup_caches(max_seq_length >= max(input_pos)+1)?")

    @torch.no_grad()
    def update(self, input_pos: Tensor, k_val: Tensor, v_val: Tensor, v_norm: Optional[Tensor] = None,
               k_hard: Optional[Tensor] = None, *, pos0: Optional[int] = None, hash_keys: bool = False):
        """Write k_val / v_val [B,S,H,D] at positions input_pos [S].

        With v_norm [B,S,H] and k_hard [B,S,H,L] given (the reference's calling
        convention) they are stored as passed; with `hash_keys=True` the codes and
        norms are computed from the rows by the fused kernel instead.  `pos0` is
        the host's copy of input_pos[0]; a decode step (S == 1) never needs it,
        a prefill without it reads it back from the device once."""
        assert input_pos.ndim == 1, f"input_pos must be [S], got {tuple(input_pos.shape)}"
        S = int(input_pos.numel())
        assert k_val.ndim == 4 and v_val.ndim == 4
        assert k_val.shape[1] == S and v_val.shape[1] == S, "k/v S dim must match input_pos length"
        if S == 0:
            return self.k_cache, self.v_cache
        if S == 1 and pos0 is None:
            # decode step: the position stays on the device.  One outside the cache
            # writes nothing (the reference raises; here the host never sees the value).
            Tcap = self.k_cache.size(2)
            pos = input_pos.long()
            ok = (pos >= 0) & (pos < Tcap)
            at = pos.clamp(0, Tcap - 1)
            for buf, val in ((self.k_cache, k_val), (self.v_cache, v_val)):
                buf.index_copy_(2, at, torch.where(ok, val.permute(0, 2, 1, 3), buf.index_select(2, at)))
            pos_b = input_pos.to(torch.int32).expand(self.lens.numel()).contiguous()
            if hash_keys:
                _hash_rows(self, k_val, v_val, pos_b=pos_b)
            elif k_hard is not None:
                raise RuntimeError("KVCache.update: precomputed k_hard needs the host position (pass pos0)")
            # the cached length follows the position (the reference masks by it every
            # step, GPT-FAST/model.py:486-487): a cache reused at an earlier position
            # does not expose the rows a longer sequence left behind
            self.lens.copy_(torch.where(ok, pos_b + 1, self.lens))
            return self.k_cache, self.v_cache
        if pos0 is not None:
            # the caller vouches for one ascending run that starts at pos0 (prefill: arange)
            self._bounds(pos0, S)
            self._write_run(pos0, k_val, v_val, v_norm, k_hard, hash_keys)
            self.lens.fill_(pos0 + S)
            return self.k_cache, self.v_cache
        # Any index tensor, as the reference's advanced-index write takes (model.py:208-226):
        # the positions come to the host once (the reference reads their extremes back too) and
        # are written as the maximal ascending runs they consist of, in order, so that a
        # position listed twice keeps its last row.
        pos = [int(p) for p in input_pos.tolist()]
        lo, hi = min(pos), max(pos)
        if lo < 0:
            self._bounds(lo, 1)
        self._bounds(hi, 1)
        start = 0
        for i in range(1, S + 1):
            if i == S or pos[i] != pos[i - 1] + 1:
                sl = slice(start, i)
                self._write_run(pos[start], k_val[:, sl], v_val[:, sl],
                                None if v_norm is None else v_norm[:, sl],
                                None if k_hard is None else k_hard[:, sl], hash_keys)
                start = i
        self.lens.fill_(hi + 1)
        return self.k_cache, self.v_cache

    @torch.no_grad()
    def update_projected(self, qkv: Tensor, freqs_cis: Tensor, n_heads: int, pos0: int, hash_keys: bool = False):
        """`update` for the projected rows qkv [B,S,(Hq+2Hkv)*D] of a prompt at pos0, with the rotary embedding
        (freqs_cis [S,D/2,2]) in the same launch; returns the rotated queries [B,S,Hq,D] and the new rows of
        keys and values as [B,S,Hkv,D] views of the cache."""
        S = qkv.shape[1]
        self._bounds(pos0, S)
        q = decode_ops.rope_rows(qkv, freqs_cis, self.k_cache, self.v_cache, pos0, n_heads, self.k_cache.size(1), self.lens)
        k, v = (c[:, :, pos0:pos0 + S].transpose(1, 2) for c in (self.k_cache, self.v_cache))
        if hash_keys:
            _hash_rows(self, k, v, t0=pos0)
        return q, k, v

    def _write_run(self, pos0: int, k_val: Tensor, v_val: Tensor, v_norm: Optional[Tensor],
                   k_hard: Optional[Tensor], hash_keys: bool) -> None:
        """Rows [pos0, pos0 + S) of every buffer from k_val / v_val [B,S,H,D]."""
        S = k_val.shape[1]
        self.k_cache[:, :, pos0:pos0 + S].copy_(k_val.permute(0, 2, 1, 3))
        self.v_cache[:, :, pos0:pos0 + S].copy_(v_val.permute(0, 2, 1, 3))
        if hash_keys:
            _hash_rows(self, k_val, v_val, t0=pos0)
        else:
            if v_norm is not None:
                self.v_norm[:, :, pos0:pos0 + S].copy_(v_norm.permute(0, 2, 1))
            if k_hard is not None:
                hash_cache.pack_codes_into(k_hard.permute(0, 2, 3, 1), self.codes, self.K, t0=pos0)


# The places where the attention hook enters the HIP library.  They are
# module-level so that a test can stand a checker in for one of them; the
# product has no other route.
def _hash_rows(cache: KVCache, k_bshd: Tensor, v_bshd: Tensor, t0: int = 0, pos_b: Optional[Tensor] = None) -> None:
    assert cache.planes_words is not None, "hash planes were not set on this cache"
    hash_cache.hash_keys_into(k_bshd, v_bshd, cache.planes_words, cache.codes, cache.v_norm, cache.L, cache.K,
                              t0=t0, pos_b=pos_b, layout="bshd")


def _sparse_is_slower(cfg: "ModelArgs", cache: KVCache, n_head: int) -> bool:
    """config.dense_below_crossover: True when a dense step over this cache is priced
    below the sparse one (decided from the cache's capacity, on the host)."""
    if not getattr(cfg, "dense_below_crossover", False) or not cache.k_cache.is_cuda:
        return False
    B, Hkv, T, D = cache.k_cache.shape
    sparse_us, dense_us = hash_cache.step_cost_estimate(
        B, n_head, Hkv, D, T, cache.L, cache.K, cache.R, int(cfg.heavy_const), int(cfg.sink_size),
        int(cfg.window_size), cache.k_cache.dtype == torch.bfloat16, cache.k_cache.element_size())
    return dense_us < sparse_us


def _sparse_step(q_bhd: Tensor, q_probs: Tensor, cache: KVCache, T: int, sink: int, window: int, M: int) -> Tensor:
    """One layer's score -> select -> attend.  Issued on the current stream; under graph
    capture the attention is the one-launch form on the library's per-GPU scratch array
    (`hash_cache.sparse_decode_step`): replays of such graphs must not overlap on a GPU."""
    return hash_cache.sparse_decode_step(q_bhd, q_probs, cache.k_cache, cache.v_cache, cache.codes, cache.v_norm,
                                         T, cache.K, sink, window, M, lens=cache.lens)


def _dense_step(q_bhd: Tensor, cache: KVCache) -> Tensor:
    return dense_decode_fwd(q_bhd, cache.k_cache, cache.v_cache, cache.lens)


def _soft_hash(q_bhd: Tensor, planes: Tensor, protos_T: Tensor, n_kv_heads: int, context_len: int = 0) -> Tensor:
    """The query's bucket probabilities, in the table layout the scorer wants for a
    context of `context_len` tokens (0: the reference's [B,H,L,R])."""
    grouped = context_len > 0 and hash_cache.prefers_grouped(q_bhd, planes, protos_T, n_kv_heads, context_len)
    return hash_cache.soft_hash(q_bhd, planes, protos_T, 1.0, n_kv_heads, grouped=grouped)


def _decode_prologue(qkv: Tensor, freqs_table: Tensor, input_pos: Tensor, cache: KVCache, planes: Tensor,
                     protos_T: Tensor, n_heads: int, n_kv_heads: int):
    """Rotary + append + hash of the new key + soft hash of the new query in one
    launch; None when the shapes are not the ones that launch is written for."""
    D = cache.k_cache.size(-1)
    if cache.planes_words is None or freqs_table.dtype not in (torch.bfloat16, torch.float32) \
            or not hash_cache.decode_prologue_fits(qkv, D, cache.K, protos_T.shape[1], n_heads, n_kv_heads,
                                                   (freqs_table, cache.k_cache, cache.v_cache, planes, protos_T)):
        return None
    T = cache.k_cache.size(2)
    grouped = hash_cache._prefers_grouped(qkv.shape[0], n_heads, n_kv_heads, T, hash_cache.dtype_enum(qkv.dtype),
                                          cache.L, cache.K, int(protos_T.shape[1]))
    return hash_cache.decode_prologue(qkv, freqs_table, input_pos, cache.k_cache, cache.v_cache, cache.lens,
                                      cache.planes_words, cache.codes, cache.v_norm, planes, protos_T, n_heads,
                                      n_kv_heads, grouped=grouped)


def _planes_to_words(planes: Tensor) -> Tensor:
    return hash_cache.permute_planes(planes)


class DecodeStep:
    """What the layers of one fused single-token step share: the rotary table and
    the token position as int32 per sequence."""
    __slots__ = ("freqs_table", "pos_b")

    def __init__(self, freqs_table: Tensor, pos_b: Tensor):
        self.freqs_table, self.pos_b = freqs_table, pos_b


class Transformer(nn.Module):
    def __init__(self, config: ModelArgs) -> None:
        super().__init__()
        self.config = config
        self.tok_embeddings = nn.Embedding(config.vocab_size, config.dim)
        self.layers = nn.ModuleList(TransformerBlock(config) for _ in range(config.n_layer))
        self.norm = RMSNorm(config.dim, eps=config.norm_eps)
        self.output = nn.Linear(config.dim, config.vocab_size, bias=False)
        self.register_buffer("freqs_cis", None, persistent=False)
        self.max_batch_size = -1
        self.max_seq_length = -1
        self.fused_decode = True     # single-token steps on the device use the fused helper kernels

    def setup_caches(self, max_batch_size, max_seq_length):
        if self.max_seq_length >= max_seq_length and self.max_batch_size >= max_batch_size:
            return
        device = self.tok_embeddings.weight.device
        dtype = self.tok_embeddings.weight.dtype
        cfg = self.config
        max_seq_length = find_multiple(max_seq_length, 8)
        self.max_seq_length = max_seq_length
        self.max_batch_size = max_batch_size
        for b in self.layers:
            b.attention.kv_cache = KVCache(max_batch_size, max_seq_length, cfg.n_local_heads, cfg.head_dim,
                                           L=cfg.L, R=cfg.R, dtype=dtype, K=cfg.K, device=device)
            b.attention.sync_planes()
        self.freqs_cis = precompute_freqs_cis(cfg.block_size, cfg.head_dim, cfg.rope_base).to(device=device)

    def step_state(self) -> list:
        """Tensors whose old contents a decode step needs again to be repeated from the same
        position.  None here: a step rewrites its own cache row and reads it back."""
        return []

    def _positions(self, idx: Tensor, input_pos: Tensor, pos0: Optional[int]):
        assert self.freqs_cis is not None, "Caches must be initialized first"
        return self._check_positions(idx, input_pos, pos0)

    def _check_positions(self, idx: Tensor, input_pos: Tensor, pos0: Optional[int]):
        """Device positions (long) and, for a prefill, the host's first position."""
        if input_pos.dtype != torch.long:
            input_pos = input_pos.long()
        S = idx.shape[1]
        if S == 1 and pos0 is None:
            return input_pos, None               # decode step: no read-back, kernels clamp by the cache's lengths
        if pos0 is None:
            pos0 = int(input_pos[0])
        if pos0 < 0 or pos0 + S > self.max_seq_length:
            raise RuntimeError(
                f"input_pos out of bounds: [{pos0},{pos0 + S - 1}] vs max_seq_length={self.max_seq_length}. "
                f"Call setup_caches(max_seq_length >= max(input_pos)+1).")
        return input_pos, pos0

    def _run(self, idx: Tensor, input_pos: Tensor, sparse: bool, pos0: Optional[int], last_only: bool,
             rows: Optional[Sequence[int]] = None) -> Tensor:
        input_pos, pos0 = self._positions(idx, input_pos, pos0)
        if idx.dtype != torch.long:
            idx = idx.long()
        x = self.tok_embeddings(idx)
        if self.fused_decode and x.is_cuda and idx.shape[1] == 1 and pos0 is None and self.layers[0].attention.kv_cache is not None:
            # one token on the device: rotary + append, norms and the SiLU product are
            # single launches; the position is handed on as it is (and once as int32
            # per sequence for the hashing kernel)
            step = DecodeStep(self.freqs_cis, input_pos.to(torch.int32).expand(idx.shape[0]).contiguous())
            # a block hands on its residual stream and its FFN output separately: their sum
            # is taken by the next norm's launch (the same add, rounded the same way)
            ffn = None
            for layer in self.layers:
                x, ffn = layer._run_fused(x, ffn, input_pos, sparse, step)
            return decode_ops.linear_rows(decode_ops.add_rmsnorm(x, self.norm.weight, self.norm.eps, residual=ffn)[1],
                                          self.output.weight)
        # (a decode step's position is unchecked on the host: keep the table lookup in range)
        freqs_cis = self.freqs_cis[input_pos if pos0 is not None else input_pos.clamp(0, self.freqs_cis.size(0) - 1)]
        ffn = None
        for layer in self.layers:
            x, ffn = layer._run_pending(x, ffn, input_pos, freqs_cis, sparse, pos0)
        pick = list(rows) if rows is not None else slice(-1, None) if last_only else slice(None)
        if rows is not None or last_only:           # (the last sum only where it is wanted)
            x, ffn = x[:, pick], None if ffn is None else ffn[:, pick]
        return self.output(_add_norm(self.norm, x, ffn)[1])

    def forward(self, idx: Tensor, input_pos: Optional[Tensor] = None, *, pos0: Optional[int] = None,
                last_only: bool = False, rows: Optional[Sequence[int]] = None) -> Tensor:
        """Dense attention everywhere (GPT-FAST/model.py:296-316).  `last_only`
        returns logits of the last position only (a long prefill needs no more),
        `rows` those of the listed places among the new tokens."""
        return self._run(idx, input_pos, False, pos0, last_only, rows)

    def sparse_forward(self, idx: Tensor, input_pos: Optional[Tensor] = None, *, pos0: Optional[int] = None,
                       last_only: bool = False) -> Tensor:
        """Hash-maintaining prefill, sparse decode (GPT-FAST/model.py:314-329)."""
        return self._run(idx, input_pos, True, pos0, last_only)

    @classmethod
    def from_name(cls, name: str):
        return cls(ModelArgs.from_name(name))


class TransformerBlock(nn.Module):
    def __init__(self, config: ModelArgs) -> None:
        super().__init__()
        self.attention = Attention(config)
        self.feed_forward = FeedForward(config)
        self.ffn_norm = RMSNorm(config.dim, config.norm_eps)
        self.attention_norm = RMSNorm(config.dim, config.norm_eps)

    def _run(self, x, input_pos, freqs_cis, sparse: bool, pos0):
        h, ffn = self._run_pending(x, None, input_pos, freqs_cis, sparse, pos0)
        return h + ffn

    def _run_pending(self, x, pending, input_pos, freqs_cis, sparse: bool, pos0):
        """The block on x + pending (None: x); returns its residual stream and its feed-forward output, not yet added."""
        x, n = _add_norm(self.attention_norm, x, pending)
        h, n = _add_norm(self.ffn_norm, x, self.attention._run(n, freqs_cis, input_pos, sparse, pos0))
        return h, self.feed_forward(n)

    def _run_fused(self, x, pending, input_pos, sparse: bool, step: "DecodeStep"):
        """One token through the block.  The block's input is x + pending (`pending`:
        the previous block's FFN output, None for the first); returns the new
        residual stream and this block's FFN output, not yet added."""
        an, fn, ff = self.attention_norm, self.ffn_norm, self.feed_forward
        # (each norm runs inside the launch of the product it feeds)
        x, qkv = decode_ops.norm_linear_rows(x, an.weight, an.eps, pending, self.attention.wqkv.weight)
        a = self.attention._run_fused_qkv(qkv, input_pos, sparse, step)
        h, g = decode_ops.norm_linear_rows(x, fn.weight, fn.eps, a, ff.w1.weight, ff.w3.weight)
        return h, decode_ops.linear_rows(g, ff.w2.weight)

    def forward(self, x: Tensor, input_pos: Tensor, freqs_cis: Tensor, mask: Tensor = None) -> Tensor:
        return self._run(x, input_pos, freqs_cis, False, None)

    def sparse_forward(self, x: Tensor, input_pos: Tensor, freqs_cis: Tensor, mask: Tensor = None) -> Tensor:
        return self._run(x, input_pos, freqs_cis, True, None)


class Attention(nn.Module):
    def __init__(self, config: ModelArgs):
        super().__init__()
        assert config.dim % config.n_head == 0
        total_head_dim = (config.n_head + 2 * config.n_local_heads) * config.head_dim
        self.wqkv = nn.Linear(config.dim, total_head_dim, bias=False)
        self.wo = nn.Linear(config.dim, config.dim, bias=False)
        self.kv_cache: Optional[KVCache] = None
        self.n_head = config.n_head
        self.head_dim = config.head_dim
        self.n_local_heads = config.n_local_heads
        self.dim = config.dim
        self._register_load_state_dict_pre_hook(self.load_hook)
        self.config = config
        self.L, self.R, self.K = config.L, config.R, config.K
        self.heavy_const = config.heavy_const
        self.register_buffer("planes", torch.randn(self.L, self.K, self.head_dim) * 0.02)
        self.register_buffer("protos_T", torch.randn(self.K, self.R) * 0.02)

    def load_hook(self, state_dict, prefix, *args):
        if prefix + "wq.weight" in state_dict:
            wq = state_dict.pop(prefix + "wq.weight")
            wk = state_dict.pop(prefix + "wk.weight")
            wv = state_dict.pop(prefix + "wv.weight")
            state_dict[prefix + "wqkv.weight"] = torch.cat([wq, wk, wv])

    def sync_planes(self) -> None:
        """Hand the current hyperplanes to the cache in the hashing kernel's
        column order; call again after changing `planes`."""
        if self.kv_cache is not None:
            self.kv_cache.planes_words = _planes_to_words(self.planes)

    # ---- hashes (GPT-FAST/model.py:392-413) ------------------------------------------
    def soft_hash(self, queries_bhd: Tensor) -> Tensor:
        """softmax_r( tanh(q . planes) / sqrt(D) @ protos_T ): [B,H,D] -> [B,H,L,R].
        One fused kernel on the device.  For tensors on the host the reference's own
        torch expression is evaluated instead: that branch exists for the host-side
        tests of the glue (tests/test_model_cpu.py) and is not a decode path -- the
        attention step itself has no host route."""
        if queries_bhd.is_cuda:
            return _soft_hash(queries_bhd, self.planes, self.protos_T, self.n_local_heads)
        proj = torch.einsum("bhd,lkd->bhlk", queries_bhd, self.planes)
        temp = max(math.sqrt(queries_bhd.size(-1)), 1e-6)
        logits = torch.einsum("bhlk,kr->bhlr", torch.tanh(proj) / temp, self.protos_T)
        return torch.softmax(logits, dim=-1)

    def pack_bits(self, bits: Tensor) -> Tensor:
        """Big-endian pack of the last dim: code = sum_k bit_k << (K-1-k), int16."""
        K = bits.shape[-1]
        weights = 1 << torch.arange(K - 1, -1, -1, device=bits.device, dtype=torch.int16)
        return (bits.to(torch.int16) * weights).sum(dim=-1).to(torch.int16)

    @torch.no_grad()
    def hard_hash_keys(self, keys_bshd: Tensor) -> Tensor:
        """int16 codes [B,S,Hkv,L] of keys [B,S,Hkv,D]: sign bits of the K
        projections of each table, zero counting as set.  On the device the
        packed words come from the hashing kernel and are unpacked into the
        reference's layout; the cache itself never takes this detour.  (Host
        tensors: the reference's einsum, for the host-side tests only.)"""
        if keys_bshd.is_cuda:
            B, S, H, _ = keys_bshd.shape
            NW = hash_cache.words_per_key(self.L, self.K)
            words = torch.empty((B, H, NW, find_multiple(S, 4)), dtype=torch.int32, device=keys_bshd.device)
            hash_cache.hash_keys_into(keys_bshd, None, _planes_to_words(self.planes), words, None, self.L, self.K,
                                      t0=0, layout="bshd")
            return hash_cache.unpack_codes(words, self.L, self.K, 0, S, layout="bthl")
        proj = torch.einsum("bshd,lkd->bshlk", keys_bshd, self.planes)
        return self.pack_bits(proj >= 0)

    # ---- the hook -------------------------------------------------------------------------
    def _run(self, x: Tensor, freqs_cis: Tensor, input_pos: Tensor, sparse: bool, pos0: Optional[int]) -> Tensor:
        bsz, seqlen, _ = x.shape
        kv_size = self.n_local_heads * self.head_dim
        qkv = self.wqkv(x)
        cache = self.kv_cache
        if seqlen > 1 and pos0 is not None and type(cache) is KVCache and decode_ops.rope_rows_fits(qkv, freqs_cis, cache.k_cache, cache.v_cache):
            # a prompt on the device: rotated and appended in one launch, attended to where it lies
            q, k, v = cache.update_projected(qkv, freqs_cis, self.n_head, pos0, hash_keys=sparse)
            return self.wo(self._prefill_attention(q, k, v, input_pos, pos0).reshape(bsz, seqlen, self.dim))
        q, k, v = qkv.split([self.dim, kv_size, kv_size], dim=-1)
        q = q.view(bsz, seqlen, self.n_head, self.head_dim)
        k = k.view(bsz, seqlen, self.n_local_heads, self.head_dim)
        v = v.view(bsz, seqlen, self.n_local_heads, self.head_dim)
        q = apply_rotary_emb(q, freqs_cis)
        k = apply_rotary_emb(k, freqs_cis)

        if sparse:
            assert cache is not None, "Call setup_caches() first so kv_cache exists"
        if cache is not None:
            cache.update(input_pos, k, v, pos0=pos0, hash_keys=sparse)

        if seqlen != 1 or cache is None:
            y = self._prefill_attention(q, k, v, input_pos, pos0)             # [B,S,H,D]
            return self.wo(y.reshape(bsz, seqlen, self.dim))

        q_bhd = q[:, 0]                                                       # [B,H,D]
        if sparse and not _sparse_is_slower(self.config, cache, self.n_head):
            T = cache.k_cache.size(2)       # upper bound; the kernels stop at cache.lens
            cfg = self.config
            # on the device the table is written in the layout the scorer prefers (same values);
            # host tensors only occur in the host-side tests, whose checker stands in for the step
            q_probs = (_soft_hash(q_bhd, self.planes, self.protos_T, self.n_local_heads, T)
                       if q_bhd.is_cuda else self.soft_hash(q_bhd))
            out_bhd = _sparse_step(q_bhd, q_probs, cache, T, int(cfg.sink_size), int(cfg.window_size),
                                   int(self.heavy_const))
        else:
            out_bhd = _dense_step(q_bhd, cache)
        return self.wo(out_bhd.reshape(bsz, 1, self.dim))

    def _run_fused(self, x: Tensor, input_pos: Tensor, sparse: bool, step: "DecodeStep") -> Tensor:
        """The decode step of `_run` with rotary embedding, K/V append and length
        update in one launch (same values)."""
        return self._run_fused_qkv(decode_ops.linear_rows(x, self.wqkv.weight), input_pos, sparse, step)

    def _run_fused_qkv(self, qkv: Tensor, input_pos: Tensor, sparse: bool, step: "DecodeStep") -> Tensor:
        """`_run_fused` from the projected row on (`qkv` = wqkv applied to the normalised input)."""
        bsz = qkv.shape[0]
        cache = self.kv_cache
        if sparse and _sparse_is_slower(self.config, cache, self.n_head):
            # below the crossover: the dense kernel, with the new key still hashed so that the
            # cache's hash state stays complete
            q_bhd, k_new, v_new = decode_ops.rope_append(qkv, step.freqs_table, input_pos, cache.k_cache,
                                                         cache.v_cache, cache.lens, self.n_head,
                                                         self.n_local_heads, return_new=True)
            _hash_rows(cache, k_new, v_new, pos_b=step.pos_b)
            out_bhd = _dense_step(q_bhd, cache)
        elif sparse:
            cfg = self.config
            fused = _decode_prologue(qkv, step.freqs_table, input_pos, cache, self.planes, self.protos_T,
                                     self.n_head, self.n_local_heads)
            if fused is not None:
                q_bhd, q_probs = fused
            else:
                q_bhd, k_new, v_new = decode_ops.rope_append(qkv, step.freqs_table, input_pos, cache.k_cache,
                                                             cache.v_cache, cache.lens, self.n_head,
                                                             self.n_local_heads, return_new=True)
                _hash_rows(cache, k_new, v_new, pos_b=step.pos_b)
                q_probs = _soft_hash(q_bhd, self.planes, self.protos_T, self.n_local_heads, cache.k_cache.size(2))
            out_bhd = _sparse_step(q_bhd, q_probs, cache, cache.k_cache.size(2), int(cfg.sink_size),
                                   int(cfg.window_size), int(self.heavy_const))
        else:
            q_bhd = decode_ops.rope_append(qkv, step.freqs_table, input_pos, cache.k_cache, cache.v_cache,
                                           cache.lens, self.n_head, self.n_local_heads)
            out_bhd = _dense_step(q_bhd, cache)
        return decode_ops.linear_rows(out_bhd.reshape(bsz, 1, self.dim), self.wo.weight)

    def _prefill_attention(self, q, k, v, input_pos, pos0) -> Tensor:
        """Causal attention of a block of new tokens over the cache prefix and
        itself (dense in both modes, as GPT-FAST/model.py:466-481)."""
        gqa = self.n_head != self.n_local_heads
        qh = q.transpose(1, 2)
        alone = self.kv_cache is None or pos0 == 0
        if not alone:
            end = pos0 + q.shape[1]
            kc, vc = self.kv_cache.k_cache[:, :, :end], self.kv_cache.v_cache[:, :, :end]
        kt, vt = (k, v) if alone else (kc.transpose(1, 2), vc.transpose(1, 2))
        if layer_ops.prompt_attend_fits(q, kt, vt) and (
                alone or layer_ops.portion_pays(q.shape[0], self.n_head, self.n_local_heads, self.head_dim, q.shape[1], kt.shape[1])):
            # (a block by itself is attended to as the library's flash kernels do it, weights in the model's
            # type unless these are switched off; over the cache the masked form kept them in 32 bits, and a token
            # sees what its position says)
            return layer_ops.prompt_attend(q, kt, vt, 0 if alone else pos0, self.head_dim ** -0.5,
                                           positions=None if alone else input_pos.contiguous(),
                                           weights16=alone and layer_ops.flash_weights())
        if alone:
            y = F.scaled_dot_product_attention(qh, k.transpose(1, 2), v.transpose(1, 2), is_causal=True,
                                               enable_gqa=gqa)
        else:
            mask = torch.arange(end, device=q.device)[None, :] <= input_pos[:, None]      # [S,end]
            y = F.scaled_dot_product_attention(qh, kc, vc, attn_mask=mask, enable_gqa=gqa)
        return y.transpose(1, 2)

    def forward(self, x: Tensor, freqs_cis: Tensor, mask: Tensor, input_pos: Optional[Tensor] = None) -> Tensor:
        """Dense attention (GPT-FAST/model.py:562-589); `mask` is accepted and unused."""
        return self._run(x, freqs_cis, input_pos.long(), False, None)

    def sparse_forward(self, x: Tensor, freqs_cis: Tensor, mask1: Tensor, mask2: Tensor,
                       input_pos: Optional[Tensor] = None) -> Tensor:
        """The SOCKET hook (GPT-FAST/model.py:415-560); the masks are accepted and unused."""
        assert input_pos is not None, "sparse_forward expects input_pos"
        return self._run(x, freqs_cis, input_pos.long(), True, None)


class FeedForward(nn.Module):
    def __init__(self, config: ModelArgs) -> None:
        super().__init__()
        self.w1 = nn.Linear(config.dim, config.intermediate_size, bias=False)
        self.w3 = nn.Linear(config.dim, config.intermediate_size, bias=False)
        self.w2 = nn.Linear(config.intermediate_size, config.dim, bias=False)

    def forward(self, x: Tensor) -> Tensor:
        a, b = self.w1(x), self.w3(x)
        if not torch.jit.is_scripting():
            if decode_ops.pointwise_fits(a, b) and a.numel() > 0 and a.shape == b.shape:
                return self.w2(decode_ops.silu_mul(a, b))
        return self.w2(F.silu(a) * b)


class RMSNorm(nn.Module):
    def __init__(self, dim: int, eps: float = 1e-5):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim))

    def forward(self, x: Tensor) -> Tensor:
        if not torch.jit.is_scripting():
            if decode_ops.pointwise_fits(x, self.weight) and x.numel() > 0 and x.shape[-1] == self.weight.numel():
                return decode_ops.add_rmsnorm(x, self.weight, self.eps)[1]
        xf = x.float()
        return (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + self.eps)).type_as(x) * self.weight

    def add(self, x: Tensor, residual: Optional[Tensor]) -> Tuple[Tensor, Tensor]:
        """(x + residual, its norm), the add and the norm by one launch where the kernel takes both."""
        if residual is None:
            return x, self(x)
        if (decode_ops.pointwise_fits(x, residual) and decode_ops.pointwise_fits(x, self.weight)
                and x.numel() > 0 and x.shape == residual.shape and x.shape[-1] == self.weight.numel()
                and type(self) is RMSNorm and "forward" not in self.__dict__ and not self._forward_hooks and not self._forward_pre_hooks
                and not nn.modules.module._has_any_global_hook()):
            return tuple(decode_ops.add_rmsnorm(x, self.weight, self.eps, residual=residual))
        h = x + residual
        return h, self(h)


def _add_norm(norm: nn.Module, x: Tensor, residual: Optional[Tensor]) -> Tuple[Tensor, Tensor]:
    """(x + residual, its norm); residual None: x.  `norm` may be any module that a caller has put there."""
    if isinstance(norm, RMSNorm):
        return norm.add(x, residual)
    h = x if residual is None else x + residual
    return h, norm(h)


def precompute_freqs_cis(seq_len: int, n_elem: int, base: float = 10000, dtype=torch.bfloat16) -> Tensor:
    """[seq_len, n_elem/2, 2] (cos, sin) table, stored in bfloat16 as
    GPT-FAST/model.py:617-623 stores it; with dtype float32 the angles are taken in
    double precision and the table rounded once."""
    if dtype == torch.float32:
        inv = float(base) ** (-torch.arange(0, n_elem, 2, dtype=torch.float64) / max(n_elem, 1))
        ang = torch.outer(torch.arange(seq_len, dtype=torch.float64), inv)
        return torch.stack([ang.cos(), ang.sin()], dim=-1).float()
    inv = 1.0 / (base ** (torch.arange(0, n_elem, 2)[: n_elem // 2].float() / n_elem))
    ang = torch.outer(torch.arange(seq_len).float(), inv)
    return torch.stack([ang.cos(), ang.sin()], dim=-1).to(torch.bfloat16)


def apply_rotary_emb(x: Tensor, freqs_cis: Tensor) -> Tensor:
    """Rotate the (2i, 2i+1) pairs of x [B,S,H,D] by the angles of freqs_cis
    [S,D/2,2], in fp32 (GPT-FAST/model.py:626-639)."""
    xs = x.float().reshape(*x.shape[:-1], -1, 2)
    fc = freqs_cis.view(1, xs.size(1), 1, xs.size(3), 2)
    re = xs[..., 0] * fc[..., 0] - xs[..., 1] * fc[..., 1]
    im = xs[..., 1] * fc[..., 0] + xs[..., 0] * fc[..., 1]
    return torch.stack([re, im], dim=-1).flatten(3).type_as(x)
