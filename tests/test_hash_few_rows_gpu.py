"""Hashing few rows (planes and keys straight into registers) against the same rows inside a call of many, bit for bit."""
import pytest
import torch

from socket_amd import hash_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"
PIECES = [(0, 1), (1, 15), (16, 17), (40, 63), (110, 65), (200, 333), (1000, 2900)]    # around 16 and 64 rows a tile


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D,L,P", [(128, 60, 10), (64, 60, 10), (40, 7, 16), (8, 9, 4), (128, 3, 10)])
def test_pieces_equal_the_whole(D, L, P, dt):
    g = torch.Generator(device=DEV).manual_seed(D + L)
    H, T = 3, 210000 // hash_cache.words_per_key(L, P) + 4000          # (three times that is past the few rows' limit)
    k = torch.randn(1, H, T, D, generator=g, device=DEV).to(dt)
    v = torch.randn(1, T, H, D, generator=g, device=DEV).to(dt).transpose(1, 2)
    words = hash_cache.permute_planes(torch.randn(L, P, D, generator=g, device=DEV))

    def fresh():
        return (torch.zeros(1, H, hash_cache.words_per_key(L, P), T, dtype=torch.int32, device=DEV),
                torch.zeros(1, H, T, dtype=torch.float16, device=DEV))

    codes, norms = fresh()
    hash_cache.hash_keys_into(k, v, words, codes, norms, L, P)
    got_codes, got_norms = fresh()
    seen = torch.zeros(T, dtype=torch.bool, device=DEV)
    for s, n in PIECES:
        hash_cache.hash_keys_into(k[:, :, s:s + n], v[:, :, s:s + n], words, got_codes, got_norms, L, P, t0=s)
        seen[s:s + n] = True
    assert torch.equal(got_codes, codes * seen) and torch.equal(got_norms, norms * seen)
    again, none = fresh()
    hash_cache.hash_keys_into(k[:, :, :77], None, words, again, None, L, P)
    assert torch.equal(again[..., :77], codes[..., :77]) and not again[..., 77:].any()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_positions_outside_the_cache_are_dropped(dt):
    g = torch.Generator(device=DEV).manual_seed(1)
    B, H, T = 37, 2, 24
    k, v = (torch.randn(B, 1, H, 128, generator=g, device=DEV).to(dt) for _ in range(2))
    words = hash_cache.permute_planes(torch.randn(60, 10, 128, generator=g, device=DEV))
    pos = torch.arange(-5, B - 5, dtype=torch.int32, device=DEV)
    codes, norms = torch.zeros(B, H, 20, T, dtype=torch.int32, device=DEV), torch.zeros(B, H, T, dtype=torch.float16, device=DEV)
    hash_cache.hash_keys_into(k, v, words, codes, norms, 60, 10, pos_b=pos, layout="bshd")
    for b in range(B):
        one, n1 = torch.zeros_like(codes[:1]), torch.zeros_like(norms[:1])
        p = int(pos[b])
        if 0 <= p < T:
            hash_cache.hash_keys_into(k[b:b + 1], v[b:b + 1], words, one, n1, 60, 10, t0=p, layout="bshd")
            assert one[0, :, :, p].any()
        assert torch.equal(codes[b], one[0]) and torch.equal(norms[b], n1[0])
