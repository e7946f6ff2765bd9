"""Index-list builder with the reference's signature, plus the sparse
flash-decode entry points re-exported as the reference's module does
(GPT-FAST/kernels/sparse.py holds both: `build_sparse_list_decode` at :16-95 and
a copy of the decode kernels at :98-329).

`build_sparse_list_decode` takes the reference's operand layout (int16 codes per
query head, [B,H,L,T]) and returns the same `(sparse_list, sparse_len)`.  The
scorer and the top-k + list assembly are HIP kernels; heavy entries are in
descending score order with equal scores ordered by ascending index.  For the
layout the HIP path is designed around (packed codes per KV head, no relayout),
use `socket_amd.hash_cache`.
"""
from __future__ import annotations

import collections
import functools
from typing import Optional

import torch

from ._lib import SOCKET_TOPK_MAX_M, check, dtype_enum, host, lib, observed, ptr, stream_ptr
from .socket_kernels import (  # noqa: F401  (re-exported, as in the reference module)
    _check_qkv,
    attention_mask_to_allowed_prob,
    sparse_attention_fwd,
    sparse_decode_stage1,
    sparse_decode_stage2,
)

_SOFT_HASH_EXT = None


def _get_soft_hash_ext():
    global _SOFT_HASH_EXT
    if _SOFT_HASH_EXT is None:
        from .soft_hash_collision_loader import load_soft_hash_collision
        _SOFT_HASH_EXT = load_soft_hash_collision(3)
    return _SOFT_HASH_EXT


# Workspaces of the selection.  The kernel wants the arrival counters at a workspace's
# head zero on entry and leaves them zero, so a workspace is zeroed once, when it is made,
# and serves every later call that cannot overlap with another user of it:
#   * eager calls: one per (device, stream, size) -- calls on one stream are ordered;
#   * calls recorded into a HIP graph: one per (device, size), made and zeroed OUTSIDE the
#     capture by the eager call of the same shape that precedes any capture (a buffer made
#     during a capture would live in that graph's private pool, be zeroed only by a
#     recorded node, and outlive the graph in this table).  Replays of graphs that hold a
#     decode step must not overlap on one GPU (hash_cache.sparse_decode_step), which is
#     what lets them share it.
# The table is bounded: the least recently used entries are dropped beyond _SELECT_WS_MAX.
_SELECT_WS = collections.OrderedDict()
_SELECT_WS_MAX = 32


def _new_workspace(device: torch.device, nbytes: int, zero_bytes: int) -> torch.Tensor:
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
    ws[:zero_bytes].zero_()
    return ws


def _select_workspace(device: torch.device, nbytes: int, zero_bytes: int) -> torch.Tensor:
    capturing = torch.cuda.is_current_stream_capturing()
    graph_key = (device.index, None, nbytes)
    if capturing:
        ws = _SELECT_WS.get(graph_key)
        if ws is None:
            # no eager call of this shape came first: a buffer of this capture's own, zeroed by a
            # recorded node on every replay, and not kept here
            return _new_workspace(device, nbytes, zero_bytes)
        _SELECT_WS.move_to_end(graph_key)
        return ws[0]
    key = (device.index, stream_ptr(device), nbytes)
    for k in (key, graph_key):
        if k not in _SELECT_WS:
            _SELECT_WS[k] = (_new_workspace(device, nbytes, zero_bytes), zero_bytes)
        _SELECT_WS.move_to_end(k)
    while len(_SELECT_WS) > _SELECT_WS_MAX:
        _SELECT_WS.popitem(last=False)
    return _SELECT_WS[key][0]


def reset_select_workspaces() -> None:
    """Zero the arrival counters of every cached workspace again.  A selection that
    was aborted mid-launch (a device error) can leave them counting; `select_list`
    calls this when the library reports a failure, and a caller who tore down a
    stream with work in flight should too."""
    if torch.cuda.is_current_stream_capturing():
        return
    for ws, zero_bytes in _SELECT_WS.values():
        ws[:zero_bytes].zero_()


def _check_budget(M: int) -> None:
    if M > SOCKET_TOPK_MAX_M:
        raise RuntimeError(f"top-k budget {M} exceeds the supported maximum {SOCKET_TOPK_MAX_M}")


def _base_width(T: int, sink: int, window: int) -> int:
    """Entries of a list's sink and window part over T positions."""
    s_e, w_e = max(0, min(sink, T)), max(0, min(window, T))
    return max(1, s_e + (T - max(T - w_e, s_e) if w_e > 0 else 0))


@functools.lru_cache(maxsize=1024)
def _select_attend_fits(B: int, H: int, D: int, T: int, width: int, dtype: torch.dtype) -> bool:
    return dtype in (torch.float32, torch.bfloat16, torch.float16) and bool(
        lib().socket_select_attend_fits(B, H, D, T, width, dtype_enum(dtype)))


def _rows_agree(scores: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, lens, budgets) -> bool:
    """Whether each row of the scores has a query of its own, rows of k / v and, where given, an int32 length and budget, all
    on one device: the one launch reads them by address, row by row of the scores."""
    B, H, _ = scores.shape
    return (q.dim() == 3 and tuple(q.shape[:2]) == (B, H) and k.dim() == 4 and k.shape == v.shape and k.shape[0] >= B
            and all(t.device == scores.device for t in (q, k, v))
            and all(t is None or (t.dtype == torch.int32 and t.device == scores.device and t.numel() == B and t.is_contiguous())
                    for t in (lens, budgets)))


def select_attend(scores: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, sink: int, window: int, M: int, *,
                  lens=None, budgets=None) -> Optional[torch.Tensor]:
    """`select_list` and the attention of q [B,H,D] over its list of rows of k / v [B,Kv,S,D] as one launch: [B,H,D], or None
    where the two are launches of their own (long rows or lists, more rows than CUs, operands that do not agree)."""
    _check_budget(int(M))
    B, H, T = scores.shape
    D = q.shape[-1]
    width = _base_width(T, sink, window) + min(int(M), T)
    if (M < 0 or sink < 0 or window < 0 or not _select_attend_fits(B, H, D, T, width, q.dtype)
            or not _rows_agree(scores, q, k, v, lens, budgets)):
        return None
    _check_qkv(q, k, v)
    assert scores.is_cuda and scores.dtype == torch.float32
    assert scores.stride(2) == 1 and scores.stride(0) == H * scores.stride(1)
    out = torch.empty((B, H, D), dtype=q.dtype, device=q.device)
    ks, vs = k.stride(), v.stride()
    check("socket_select_attend", lib().socket_select_attend(
        ptr(scores), scores.stride(1), ptr(lens), ptr(budgets), T, int(M), int(sink), int(window), width, ptr(q), ptr(k), ptr(v),
        dtype_enum(q.dtype), q.stride(0), q.stride(1), ks[0], ks[1], ks[2], vs[0], vs[1], vs[2], ptr(out), H * D, D,
        B, H, k.shape[1], D, k.shape[2], stream_ptr(q.device)))
    return out


def select_list(scores: torch.Tensor, sink: int, window: int, M: int, *, lens=None, budgets=None,
                write_base: bool = True, list_width=None, row_range=None, split: bool = True):
    """Top-M + [sink | window | heavy] assembly on fp32 score rows [B,H,T]
    (row pitch = scores.stride(1)).  Returns (sparse_list int32 [B,H,width],
    sparse_len int32 [B,H]).  `lens`/`budgets`: optional int32 [B] device tensors
    (per-sequence context length and top-k budget).  `row_range`: the int32
    [B,H,parts,2] key ranges `hash_cache.score_packed(..., with_range=True)`
    returns for these scores (saves the kernel's first pass).  `split=False`
    keeps every row to one workgroup (the result is the same)."""
    assert scores.is_cuda and scores.dtype == torch.float32 and scores.dim() == 3
    assert scores.stride(2) == 1 and scores.stride(0) == scores.shape[1] * scores.stride(1)
    B, H, T = scores.shape
    M = int(M)
    _check_budget(M)
    if list_width is None:
        list_width = (_base_width(T, sink, window) if write_base else 0) + min(M, T)
    sparse_list = torch.empty((B, H, list_width), dtype=torch.int32, device=scores.device)
    sparse_len = torch.empty((B, H), dtype=torch.int32, device=scores.device)
    if list_width == 0:
        return sparse_list, sparse_len.zero_()
    _select_into(scores, sink, window, M, lens, budgets, write_base, row_range, split, sparse_list, sparse_len)
    return sparse_list, sparse_len


def _workspace_of(device, B: int, H: int, T: int, M: int):
    """(workspace, its bytes) of a selection: (None, 0) where every row is one workgroup's."""
    L = lib()
    nbytes = L.socket_select_workspace_bytes(B, H, T, M)
    return (_select_workspace(device, nbytes, L.socket_select_workspace_zero_bytes(B, H, T, M)) if nbytes else None), nbytes


def _select_into(scores, sink: int, window: int, M: int, lens, budgets, write_base: bool, row_range, split: bool,
                 sparse_list: torch.Tensor, sparse_len: torch.Tensor) -> None:
    """The selection's launch into the rows of `sparse_list` [B,H,width] (any stride between rows)."""
    B, H, T = scores.shape
    width = sparse_list.shape[2]
    assert sparse_list.stride(2) == 1 and sparse_list.stride(0) == H * sparse_list.stride(1)
    ws, ws_bytes = _workspace_of(scores.device, B, H, T, M) if split else (None, 0)
    try:
        check("socket_select_list", lib().socket_select_list(
            ptr(scores), scores.stride(1), ptr(lens), ptr(budgets), ptr(row_range),
            0 if row_range is None else row_range.shape[2], B, H, T, M, int(sink), int(window),
            1 if write_base else 0, ptr(sparse_list), sparse_list.stride(1), width, ptr(sparse_len),
            ptr(ws), ws_bytes, stream_ptr(scores.device)))
    except RuntimeError:
        if ws is not None:
            reset_select_workspaces()
        raise


# Entries of a row's sink and window from which they are a launch of their own, dealt out over several workgroups.  In
# the selection's launch one workgroup of a row writes them: no launch more, but 25 us per 100000 entries.  The whole operator
# over four small tables, us, in the selection's launch / in its own: 32 rows, 16000 entries 21.3 / 22.4, 32768 25.1 / 23.0, 100000 61
# / 39; 4 rows, 16000 20.1 / 21.7, 32768 23.8 / 21.2, 100000 41 / 25; 128 rows, 16000 33.6 / 36.2, 32768 39.6 / 37.8.
# The native step knows the first alone, and takes calls below here.
_LONG_BASE = 24576


def _build_in_place(q_probs, k_hard, v_norm, allowed, sink: int, window: int, M: int):
    """`build_sparse_list_decode` in two launches: scores from the operands in their own types, and the list (three where
    the window is long).  None for operands it does not take."""
    B, H, L, R = q_probs.shape
    T = k_hard.shape[3]
    types = (torch.float16, torch.bfloat16, torch.float32)
    if (min(B, H, T, L, R, M) < 1 or B * H > 65535 or v_norm.dtype not in types or k_hard.dtype != torch.int16
            or tuple(k_hard.shape[:2]) != (B, H) or tuple(v_norm.shape) != (B, H, T) or tuple(allowed.shape) != (B, H, T)
            or not all(t.device == q_probs.device for t in (k_hard, v_norm, allowed))):
        return None
    _check_budget(M)
    q_probs, k_hard, v_norm, allowed = (t.contiguous() for t in (q_probs, k_hard, v_norm, allowed))
    sink, window = max(0, min(sink, T)), max(0, min(window, T))
    base = max(1, sink + (T - max(T - window, sink) if window > 0 else 0))
    scores = torch.empty((B, H, T), dtype=torch.float32, device=q_probs.device)
    sparse_list = torch.empty((B, H, base + M), dtype=torch.int32, device=q_probs.device)
    sparse_len = torch.empty((B, H), dtype=torch.int32, device=q_probs.device)
    s = stream_ptr(q_probs.device)
    check("socket_soft_hash_collision", lib().socket_soft_hash_collision_typed(
        ptr(q_probs), dtype_enum(q_probs.dtype), ptr(k_hard), ptr(allowed), ptr(v_norm), dtype_enum(v_norm.dtype), ptr(scores),
        B, H, L, R, T, s))
    if base > _LONG_BASE:
        _select_into(scores, 0, 0, M, None, None, False, None, True, sparse_list[:, :, base:], sparse_len)
        check("socket_finish_list", lib().socket_finish_list(ptr(sparse_list), ptr(sparse_len), ptr(allowed), B * H, T, sink,
                                                             window, M, s))
        return sparse_list, sparse_len
    ws, ws_bytes = _workspace_of(scores.device, B, H, T, M)
    try:
        check("socket_select_list", lib().socket_select_list_allowed(
            ptr(scores), T, ptr(allowed), B, H, T, M, sink, window, ptr(sparse_list), base + M, base + M, ptr(sparse_len),
            ptr(ws), ws_bytes, s))
    except RuntimeError:
        if ws is not None:
            reset_select_workspaces()
        raise
    return sparse_list, sparse_len


def build_sparse_list_decode(
    q_probs: torch.Tensor,       # [B,H,L,R] fp16/bf16/fp32
    k_hard_bhlt: torch.Tensor,   # [B,H,L,T] int16/int32
    v_norm_bht: torch.Tensor,    # [B,H,T] fp16/bf16/fp32
    allowed_bht: torch.Tensor,   # [B,H,T] bool
    sink: int,
    window: int,
    M: int,
    KC: int = 8,
    BLOCK_N: int = 512,
    num_warps: int = 8,
    num_stages: int = 2,
):
    """GPT-FAST/kernels/sparse.py:16-95.  KC, BLOCK_N, num_warps, num_stages are
    accepted and ignored, as in the reference (:38)."""
    if type(q_probs) is torch.Tensor and q_probs.is_cuda and k_hard_bhlt.dtype is torch.int16 and not observed():
        # (the usual operands in one step; what it does not take is looked over here)
        built = host().build_list(q_probs, k_hard_bhlt, v_norm_bht, allowed_bht, sink, window, M, _LONG_BASE - 1, SOCKET_TOPK_MAX_M,
                                  _select_workspace, stream_ptr(q_probs.device))
        if built is not None:
            if type(built[0]) is str:
                reset_select_workspaces()
                check(*built)
            return built
    assert q_probs.is_cuda and k_hard_bhlt.is_cuda and v_norm_bht.is_cuda and allowed_bht.is_cuda
    assert q_probs.dtype in (torch.float16, torch.bfloat16, torch.float32)
    assert allowed_bht.dtype == torch.bool
    _, _, L, _ = q_probs.shape
    _, _, L2, T = k_hard_bhlt.shape
    assert L2 == L
    M_eff = min(M, T)
    built = _build_in_place(q_probs, k_hard_bhlt if k_hard_bhlt.dtype == torch.int16 else k_hard_bhlt.to(torch.int16),
                            v_norm_bht, allowed_bht, int(sink), int(window), int(M_eff))
    if built is not None:
        return built
    with torch.no_grad():
        return _build_with_torch(q_probs, k_hard_bhlt, v_norm_bht, allowed_bht, sink, window, M_eff)


def _build_with_torch(q_probs, k_hard_bhlt, v_norm_bht, allowed_bht, sink: int, window: int, M_eff: int):
    """The same with torch's operations around the scorer and the top-k, for operands `_build_in_place` does not take."""
    B, H = q_probs.shape[:2]
    T, device = k_hard_bhlt.shape[3], q_probs.device
    if M_eff > 0:
        ext = _get_soft_hash_ext()
        q_probs_f32 = q_probs.float().unsqueeze(2).contiguous()
        key_buckets = k_hard_bhlt if k_hard_bhlt.dtype == torch.int16 else k_hard_bhlt.to(torch.int16)
        key_buckets = key_buckets.contiguous()
        allowed_ext = allowed_bht.unsqueeze(2).contiguous()
        v_hist = v_norm_bht.float().unsqueeze(2).contiguous()
        scores = ext.soft_hash_collision(q_probs_f32, key_buckets, allowed_ext, v_hist).squeeze(2)
        heavy_idx, _ = select_list(scores, 0, 0, M_eff, write_base=False)
        # disallowed positions carry -inf and may still be selected when fewer
        # than M_eff positions are allowed: they become -1 (:62-68)
        ok = torch.gather(allowed_bht, -1, heavy_idx.clamp(0, T - 1).long())
        heavy_idx = heavy_idx.masked_fill(~ok, -1)
    else:
        heavy_idx = torch.empty((B, H, 0), device=device, dtype=torch.int32)

    sink = max(0, min(sink, T))
    window = max(0, min(window, T))
    parts = []
    if sink > 0:
        parts.append(torch.arange(sink, device=device, dtype=torch.int32))
    if window > 0:
        win_start = max(T - window, sink)
        if win_start < T:
            parts.append(torch.arange(win_start, T, device=device, dtype=torch.int32))
    base = torch.cat(parts, dim=0) if parts else torch.tensor([T - 1], device=device, dtype=torch.int32)
    base = base.view(1, 1, -1).expand(B, H, -1)
    base_ok = torch.gather(allowed_bht, -1, base.long())
    base = base.masked_fill(~base_ok, -1)

    sparse_list = torch.cat([base, heavy_idx], dim=-1).contiguous()
    sparse_len = torch.full((B, H), sparse_list.shape[-1], device=device, dtype=torch.int32)
    return sparse_list, sparse_len
