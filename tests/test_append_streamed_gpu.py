"""Appends large enough to stream past the planes (tiles of 64 and 128 keys, every type) against the same tokens appended a
few at a time, bit for bit."""
import pytest
import torch

from socket_amd import hash_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,S,H,D,L,P,pos0", [
    (1, 256, 8, 64, 60, 10, 3),          # the fewest rows of 64 dims, whole tiles
    (3, 129, 6, 64, 9, 4, 0),            # one row past two tiles, two words
    (1, 832, 8, 128, 60, 10, 1),         # the fewest of 128 dims with 20 words
    (2, 769, 5, 128, 72, 10, 2),         # one row past twelve tiles, 24 words, the most
    (1, 1727, 3, 128, 3, 10, 5),         # a single word; one row short of a tile
    (2, 4100, 4, 128, 32, 8, 0),         # a tile of 128 for every CU
    (1, 11003, 3, 64, 60, 10, 7),
])
def test_streamed_append_equals_small_ones(B, S, H, D, L, P, pos0, dt):
    g = torch.Generator(device=DEV).manual_seed(S + D)
    planes = torch.randn(L, P, D, generator=g, device=DEV).to(dt)
    k = torch.randn(B, S, H, D, generator=g, device=DEV).to(dt)
    v = torch.randn(B, S, 3 * H * D, generator=g, device=DEV).to(dt)[..., H * D:2 * H * D].view(B, S, H, D)

    def fresh():
        cache = hash_cache.SocketHashCache(B, pos0 + S + 5, H, D, L, P, dtype=dt, device=DEV)
        cache.set_planes(planes)
        cache.codes.fill_(77)
        return cache

    whole, parts = fresh(), fresh()
    whole.append(pos0, k, v)
    step = 2040 // (B * H)               # (below every line from which on rows are streamed)
    for s in range(0, S, step):
        parts.append(pos0 + s, k[:, s:s + step], v[:, s:s + step])
    for name in ("k_cache", "v_cache", "codes", "v_norm", "lens"):
        assert torch.equal(getattr(whole, name), getattr(parts, name)), name
    # hashed alone, without values, from the cache's rows
    codes = torch.full_like(whole.codes, 77)
    norms = torch.zeros_like(whole.v_norm)
    hash_cache.hash_keys_into(whole.k_cache[:, :, pos0:pos0 + S], None, whole.planes_words, codes, norms, L, P, t0=pos0)
    assert torch.equal(codes, whole.codes) and not norms.any()


def test_launches_follow_the_current_stream():
    """The handle the launches are given is that of torch's current stream, by tensor device, by bare device and by default;
    rows that require gradients are appended like any others."""
    from socket_amd._lib import stream_ptr
    side = torch.cuda.Stream()
    for s in (torch.cuda.current_stream(), side):
        with torch.cuda.stream(s):
            for d in (torch.zeros(1, device=DEV).device, torch.device(DEV), None):
                assert (stream_ptr(d) or 0) == s.cuda_stream
    k, v = (torch.randn(2, 9, 3, 64, device=DEV) for _ in range(2))
    caches = [hash_cache.SocketHashCache(2, 16, 3, 64, 12, 4, dtype=torch.float32, device=DEV) for _ in range(2)]
    planes = torch.randn(12, 4, 64, device=DEV)
    for cache, grad in zip(caches, (False, True)):
        cache.set_planes(planes)
        cache.append(2, k.clone().requires_grad_(grad), v)
    for name in ("k_cache", "v_cache", "codes", "v_norm", "lens"):
        assert torch.equal(getattr(caches[0], name), getattr(caches[1], name)) and not getattr(caches[1], name).requires_grad
