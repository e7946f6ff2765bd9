"""SocketHashCache.append (rows copied and hashed by one call of the library) against torch's copies and the hash
of the rows padded to 128 dims, bit for bit."""
import pytest
import torch

from socket_amd import hash_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"


def separate(cache, pos0, k, v):
    """The same cache filled by torch's copies, and codes and norms of zero-padded rows."""
    B, S, H, D = k.shape
    kc, vc, codes, norms = (t.clone() for t in (cache.k_cache, cache.v_cache, cache.codes, cache.v_norm))
    kc[:, :, pos0:pos0 + S] = k.permute(0, 2, 1, 3)
    vc[:, :, pos0:pos0 + S] = v.permute(0, 2, 1, 3)
    pad = lambda x: torch.nn.functional.pad(x, (0, 128 - D))
    hash_cache.hash_keys_into(pad(k), pad(v), cache.planes_words, codes, norms, cache.L, cache.P, t0=pos0, layout="bshd")
    return kc, vc, codes, norms


# (S of 4100 in 8 rows is past a 128-key tile per CU, the streamed launch; 40 dims are three whole MFMA steps less a
# half, 20 are no whole 16-byte pieces in 16 bits and stay with torch's copies; from some 3300 rows on, up to 13000, the
# launch without LDS takes 64 of them at a time, 64-row tiles that cross from head to head among them; 160004 float32
# rows of 128 are past the 128 MB from which the hash reads the cache)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,S,H,D,pos0", [(2, 1, 3, 128, 7), (1, 63, 2, 64, 0), (3, 129, 2, 40, 5), (1, 4100, 8, 128, 3),
                                          (2, 4097, 4, 64, 1), (2, 70, 2, 20, 2), (2, 777, 8, 64, 1003), (3, 401, 3, 40, 2),
                                          (2, 401, 7, 128, 3), (1, 40001, 4, 128, 5)])
def test_append_equals_copies_and_hash(B, S, H, D, pos0, dt):
    g = torch.Generator(device=DEV).manual_seed(S + D)
    cache = hash_cache.SocketHashCache(B, pos0 + S + 9, H, D, 60, 10, dtype=dt, device=DEV)
    cache.set_planes(torch.randn(60, 10, D, generator=g, device=DEV).to(dt))
    for t in (cache.k_cache, cache.v_cache):
        t.normal_(generator=g)
    k = torch.randn(B, S, H, D, generator=g, device=DEV).to(dt)
    v = torch.randn(B, S, 3 * H * D, generator=g, device=DEV).to(dt)[..., H * D:2 * H * D].view(B, S, H, D)
    want = separate(cache, pos0, k, v)
    assert cache._append_fits(k, v) == (D != 20 or dt == torch.float32 and D % 8 == 0)
    cache.append(pos0, k, v)
    for got, w in zip((cache.k_cache, cache.v_cache, cache.codes, cache.v_norm), want):
        assert torch.equal(got, w)
    assert (cache.lens == pos0 + S).all()
    with pytest.raises(RuntimeError):
        cache.append(cache.Tcap - S + 1, k, v)


@pytest.mark.parametrize("D", [8, 64])
def test_step_hash_of_narrow_heads(D):
    """One row per sequence at a device-side position, as a decode step hashes it; odd strides take the padded copy."""
    g = torch.Generator(device=DEV).manual_seed(D)
    k, v = (torch.randn(3, 1, 4, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    words = hash_cache.permute_planes(torch.randn(60, 10, D, generator=g, device=DEV))
    pos = torch.tensor([0, 5, 15], dtype=torch.int32, device=DEV)
    pad = lambda x: torch.nn.functional.pad(x, (0, 128 - D))
    odd = [torch.zeros(3, 1, 4, D + 1, device=DEV).bfloat16()[..., :D] for _ in range(2)]
    odd[0].copy_(k)
    odd[1].copy_(v)
    got = []
    for a, b in ((k, v), (pad(k), pad(v)), odd):
        codes = torch.zeros(3, 4, 20, 16, dtype=torch.int32, device=DEV)
        norms = torch.zeros(3, 4, 16, dtype=torch.float16, device=DEV)
        hash_cache.hash_keys_into(a, b, words, codes, norms, 60, 10, pos_b=pos, layout="bshd")
        got.append((codes, norms))
    for other in got[1:]:
        assert torch.equal(got[0][0], other[0]) and torch.equal(got[0][1], other[1])
