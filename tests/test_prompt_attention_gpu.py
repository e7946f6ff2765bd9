"""The matrix-core prompt attention of csrc/prompt_attend.hip (head widths 64 and 128, 128 + 64 shared)
against a float64 softmax at the sizes where it can go wrong: one row, the edges of a wave's 32 rows, a
workgroup's 128 rows and a tile's 64 keys, chunk borders inside a tile, keys from the ring."""
import math

import pytest
import torch

from socket_amd import layer_ops
from socket_amd.sequence_state import ChunkRing

pytestmark = pytest.mark.gpu
DEV = "cuda"


def softmax_attention(q, k, v, pos0, chunk, scale, cap=0.0):
    """float64; q [B,T,H,d] at pos0 .., k [B,S,G,d], v [B,S,G,dv] of every position."""
    rep = q.shape[2] // k.shape[2]
    k, v = k.double().repeat_interleave(rep, 2), v.double().repeat_interleave(rep, 2)
    s = torch.einsum("bthd,bshd->bhts", q.double(), k) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    i = torch.arange(pos0, pos0 + q.shape[1], device=q.device)[:, None]
    j = torch.arange(k.shape[1], device=q.device)[None]
    s = s.masked_fill((j > i) | (j < i // chunk * chunk), -math.inf)
    return torch.einsum("bhts,bshd->bthd", torch.softmax(s, -1), v)


def close(got, want, unit):
    """Rounding of the result (half a unit in the last place of its type) and as much again for the products."""
    err = (got.double() - want).norm() / want.norm()
    assert err < unit, float(err)
    assert (got.double() - want).abs().max() < 4 * unit * want.abs().max()


@pytest.mark.parametrize("T,first,H,G,D,cap", [(1, 0, 4, 2, 128, 0.0), (31, 0, 8, 2, 64, 20.0), (33, 1, 4, 4, 128, 30.0),
                                               (129, 64, 6, 2, 128, 0.0), (190, 70, 7, 1, 64, 0.0), (321, 100, 4, 1, 128, 15.0)])
def test_portions_inside_chunks(T, first, H, G, D, cap):
    """A first portion of `first` tokens fills the ring, the second of T tokens reads it; chunks of 150."""
    g = torch.Generator(device=DEV).manual_seed(T)
    chunk, n = 150, first + T
    q, k, v = (torch.randn(2, n, h, D, generator=g, device=DEV).bfloat16() for h in (H, G, G))
    ring = ChunkRing(2, n, G, D, chunk, torch.bfloat16, DEV)
    want = softmax_attention(q, k, v, 0, chunk, 0.3 * D ** -0.5, cap)
    parts = []
    for t0, t1 in ((0, first), (first, n)):
        if t1 > t0:
            parts.append(layer_ops.chunk_attend(q[:, t0:t1], k[:, t0:t1], v[:, t0:t1], ring, t0, 0.3 * D ** -0.5, cap))
    close(torch.cat(parts, 1), want, 2 ** -8)


@pytest.mark.parametrize("T,first", [(1, 3), (64, 0), (127, 1), (128, 0), (200, 61)])
def test_shared_key_segment_and_gate(T, first):
    g = torch.Generator(device=DEV).manual_seed(T)
    B, H, S = 2, 3, first + T
    q = torch.randn(B, T, H, 192, generator=g, device=DEV).bfloat16()
    kv = torch.randn(B, S, H, 256, generator=g, device=DEV).bfloat16()
    shared = torch.randn(B, S, 64, generator=g, device=DEV).bfloat16()
    gate = torch.randn(B, T, H * 128, generator=g, device=DEV).bfloat16()
    k, v = kv[..., :128], kv[..., 128:]
    got = layer_ops.causal_attend(q, k, shared, v, first, 192 ** -0.5, gate)
    want = softmax_attention(q, torch.cat([k, shared[:, :, None].expand(B, S, H, 64)], -1), v, first, 1 << 30, 192 ** -0.5)
    close(got, want * torch.sigmoid(gate.double()).view(B, T, H, 128), 2 ** -8)


def test_scores_of_any_size():
    """Rows of equal large scores, growing maxima and scores past the fp32 exponent's reach."""
    B, T, D = 1, 200, 128
    for gain in (1e-3, 30.0, 1e4, 3e8):
        g = torch.Generator(device=DEV).manual_seed(7)
        q = (torch.randn(B, T, 2, D, generator=g, device=DEV) * gain).bfloat16()
        k = (torch.randn(B, T, 2, D, generator=g, device=DEV) * torch.linspace(0.1, 3, T, device=DEV)[:, None, None]).bfloat16()
        v = torch.randn(B, T, 2, D, generator=g, device=DEV).bfloat16()
        got = layer_ops.chunk_attend(q, k, v, ChunkRing(B, T, 2, D, T, torch.bfloat16, DEV), 0, 1.0, 0.0)
        assert torch.isfinite(got).all()
        close(got, softmax_attention(q, k, v, 0, T, 1.0), 2 ** -8 if gain < 1e3 else 2 ** -6)


@pytest.mark.parametrize("B,T,first,H,G,D,dt,w16", [
    (2, 65, 0, 8, 2, 128, torch.bfloat16, True), (1, 257, 0, 6, 6, 64, torch.float16, True), (1, 128, 190, 4, 1, 128, torch.float16, False),
    (3, 2, 63, 8, 8, 64, torch.bfloat16, False), (2, 300, 37, 7, 7, 128, torch.bfloat16, False)])
def test_causal_over_a_cache(B, T, first, H, G, D, dt, w16):
    """Keys and values as a cache holds them ([B,G,S,D]), the portion's positions given or counted."""
    g = torch.Generator(device=DEV).manual_seed(T)
    q = torch.randn(B, T, H, D, generator=g, device=DEV).to(dt)
    k, v = (torch.randn(B, G, first + T + 5, D, generator=g, device=DEV).to(dt)[:, :, :first + T].transpose(1, 2) for _ in range(2))
    assert layer_ops.prompt_attend_fits(q, k, v)
    want = softmax_attention(q, k, v, first, 1 << 30, D ** -0.5)
    unit = 2 ** -8 if dt == torch.bfloat16 else 2 ** -11
    close(layer_ops.prompt_attend(q, k, v, first, D ** -0.5, weights16=w16), want, unit)
    pos = torch.arange(first, first + T, device=DEV)
    close(layer_ops.prompt_attend(q, k, v, first, D ** -0.5, pos, w16), want, unit)


def test_positions_that_are_no_run():
    """A token sees the keys up to its own position, wherever it stands; none for a position before the first."""
    g = torch.Generator(device=DEV).manual_seed(3)
    T, first, H, D = 150, 40, 4, 64
    q = torch.randn(1, T, H, D, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(1, first + T, H, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    pos = torch.randint(0, first + T + 20, (T,), generator=g, device=DEV)
    got = layer_ops.prompt_attend(q, k, v, first, 0.1, pos)
    s = torch.einsum("bthd,bshd->bhts", q.double(), k.double()) * 0.1
    s = s.masked_fill(torch.arange(first + T, device=DEV)[None] > pos[:, None], -math.inf)
    close(got, torch.einsum("bhts,bshd->bthd", torch.softmax(s, -1), v.double()), 2 ** -8)
    pos[7] = -1
    assert (layer_ops.prompt_attend(q, k, v, first, 0.1, pos)[:, 7] == 0).all()


def test_what_it_leaves_to_the_library():
    q = torch.randn(1, 8, 4, 64, device=DEV).bfloat16()
    assert layer_ops.prompt_attend_fits(q, q, q)
    assert not layer_ops.prompt_attend_fits(q.float(), q.float(), q.float())
    assert not layer_ops.prompt_attend_fits(q[..., :40], q[..., :40], q[..., :40])
    assert not layer_ops.prompt_attend_fits(q, q[:, :, :3], q[:, :, :3])
    assert not layer_ops.prompt_attend_fits(q[..., 1:], q[..., 1:], q[..., 1:])
    grad = q.clone().requires_grad_()
    assert not layer_ops.prompt_attend_fits(grad, q, q)
    with torch.no_grad():
        assert layer_ops.prompt_attend_fits(grad, q, q)
    seen = []
    torch.vmap(lambda x: (seen.append(layer_ops.prompt_attend_fits(x, x, x)), x)[1])(q[None])
    with torch.autograd.forward_ad.dual_level():
        seen.append(layer_ops.prompt_attend_fits(q, q, q))
    assert seen == [False, False]
