"""The scorer's launch for few tokens per CU (one or two tokens to a lane) at the edges of its tiles, slices and rules."""
import pytest
import torch

from oracle import socket_oracle as orc
from socket_amd import hash_cache
from socket_amd._lib import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hkv,G,L,P,T,dt", [
    (1, 1, 4, 60, 10, 1, torch.float32),             # one token
    (2, 2, 2, 3, 10, 63, torch.bfloat16),            # one packed word, less than a wave
    (1, 8, 4, 60, 10, 4097, torch.float32),          # one word to a slice
    (1, 8, 4, 60, 10, 32768, torch.bfloat16),        # a full tile for every CU
    (1, 8, 4, 60, 10, 32771, torch.bfloat16),        # a second token for one wave of a tile
    (1, 8, 4, 57, 10, 40003, torch.float32),         # a second token for some waves, an odd number of words
    (3, 4, 7, 48, 10, 5001, torch.bfloat16),         # two parts of a group, rows that are no divisor of 8
    (2, 4, 7, 28, 8, 16333, torch.float32),          # slices of three words, a short last one
    (2, 8, 2, 80, 8, 12345, torch.bfloat16),         # twenty words, slices of twelve
    (5, 1, 8, 32, 8, 259, torch.float32),
])
def test_scores_of_few_tokens_per_cu(B, Hkv, G, L, P, T, dt):
    """Equal to the definition (bit for bit with an fp32 table, 2e-6 where the matrix core adds bf16 entries) with and
    without the fill, for sequences of length 0, 1, around a wave and as long as the context; and to the other launches."""
    dev, R, Hq = "cuda", 1 << P, Hkv * G
    assert lib().socket_score_lanes_serve(B, Hq, Hkv, T, 0 if dt == torch.float32 else 1, L, P, R) == 1
    g = torch.Generator(device=dev).manual_seed(T)
    qp = (torch.rand(B, Hq, L, R, generator=g, device=dev) * torch.exp(-8 * torch.rand(B, Hq, L, R, generator=g, device=dev))).to(dt)
    codes = torch.randint(0, R, (B, Hkv, L, T), generator=g, device=dev, dtype=torch.int32).to(torch.int16)
    Tcap = (T + 7) // 8 * 8
    packed = torch.zeros(B, Hkv, orc.words_per_key(L, P), Tcap, dtype=torch.int32, device=dev)
    hash_cache.pack_codes_into(codes, packed, P, t0=0)
    vn = torch.zeros(B, Hkv, Tcap, dtype=torch.float16, device=dev)
    vn[..., :T] = (torch.rand(B, Hkv, T, generator=g, device=dev) * 6).half()
    want = torch.zeros(B, Hq, T, device=dev)
    where = codes.long().repeat_interleave(G, 1)
    for l in range(L):
        want += torch.gather(qp[:, :, l].float(), 2, where[:, :, l])
    want *= vn[..., :T].float().repeat_interleave(G, 1)
    table, tol = hash_cache.group_q_probs(qp, Hkv), 0.0 if dt == torch.float32 else 2e-6
    pool = [T, 0, 1, T // 2 + 1, min(T, 65)]
    for lens in (None, torch.tensor([min(T, pool[b % len(pool)]) for b in range(B)], dtype=torch.int32, device=dev)):
        n = torch.full((B,), T, device=dev) if lens is None else lens
        hidden = torch.arange(T, device=dev)[None, None] >= n[:, None, None]
        ref = want.masked_fill(hidden, float("-inf"))
        got = hash_cache.score_packed(table, packed, vn, T, P, lens=lens, n_heads=Hq)
        assert torch.equal(torch.isinf(got), torch.isinf(ref))
        assert ((got - ref).abs() / ref.abs().clamp_min(1e-30)).nan_to_num(0).max().item() <= tol
        out = torch.full((B, Hq, (T + 3) // 4 * 4), 123.0, device=dev)
        rows = hash_cache.score_packed(table, packed, vn, T, P, lens=lens, n_heads=Hq, out=out, skip_masked=True)
        assert torch.equal(rows[~hidden.expand_as(rows)], got[~hidden.expand_as(rows)])
        assert (rows[hidden.expand_as(rows)] == 123.0).all() and (out[:, :, T:] == 123.0).all()
        tiled, _ = hash_cache.score_packed(table, packed, vn, T, P, lens=lens, n_heads=Hq, with_range=True)
        assert ((got - tiled).abs() / tiled.abs().clamp_min(1e-30)).nan_to_num(0).max().item() <= tol
