"""The matrix-core soft hash (bf16, 128 dims, K = 10, R = 1024) against float64: every width of a unit, padded groups, units
that do not fill a workgroup's sixteen heads, both output types, and one head's NaN kept to itself."""
import math

import pytest
import torch

from socket_amd import hash_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"


def exact(q, planes, protos, temperature):
    t = torch.tanh(torch.einsum("bhd,lkd->bhlk", q.double(), planes.double())) / math.sqrt(q.shape[-1])
    return torch.softmax(torch.einsum("bhlk,kr->bhlr", t, protos.double()) / temperature, -1)


def inputs(B, Hq, L, seed, cube):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = torch.randn(B, Hq, 128, generator=g, device=DEV).bfloat16()
    planes = (torch.randn(L, 10, 128, generator=g, device=DEV) * (1.0 if cube else 0.1)).bfloat16()
    r, k = torch.arange(1024, device=DEV)[None], torch.arange(10, device=DEV)[:, None]
    protos = (((r >> (9 - k)) & 1) * 2 - 1).bfloat16() if cube else torch.randn(10, 1024, generator=g, device=DEV).bfloat16()
    return q, planes, protos


@pytest.mark.parametrize("B,Hq,Hkv,L,cube,temp", [(1, 1, 1, 1, True, 0.3), (3, 6, 3, 5, False, 0.3), (1, 28, 4, 3, True, 0.3),
                                                  (2, 15, 5, 4, False, 1.0), (5, 40, 8, 2, True, 1.0), (1, 7, 7, 3, False, 0.02)])
def test_tables_of_every_layout(B, Hq, Hkv, L, cube, temp):
    q, planes, protos = inputs(B, Hq, L, B + Hq, cube)
    want = exact(q, planes, protos, temp)
    parts, width = hash_cache.group_shape(Hq, Hkv)
    G = Hq // Hkv
    plain = hash_cache.soft_hash(q, planes, protos, temp, Hkv)
    wide = hash_cache.soft_hash(q, planes, protos, temp, Hkv, out_dtype=torch.float32)
    # (ten fp32 products and sums of logits up to 0.9 / temp, an exponential and a normalisation to an ulp or two)
    unit = 2 ** -23 * (16 + 16 * 0.9 / temp)
    assert ((wide.double() - want).abs() <= unit * want).all()
    # (bfloat16 has eight significant bits: a rounding is off by up to 2^-8 of its result)
    assert ((plain.double() - want).abs() <= (2 ** -8 + 2 * unit) * want).all()
    for got, flat in ((hash_cache.soft_hash(q, planes, protos, temp, Hkv, grouped=True), plain),
                      (hash_cache.soft_hash(q, planes, protos, temp, Hkv, out_dtype=torch.float32, grouped=True), wide)):
        for h in range(Hq):
            kv, g = h // G, h % G
            assert torch.equal(got[:, kv * parts + g // width, :, :, g % width], flat[:, h])
        for g in range(G, parts * width):
            assert (got.view(B, Hkv, parts, L, 1024, width)[:, :, g // width, :, :, g % width] == 0).all()
    assert torch.equal(plain, hash_cache.soft_hash(q, planes, protos, temp, None))


def test_a_head_of_nan_stays_alone():
    q, planes, protos = inputs(2, 8, 2, 1, True)
    clean = hash_cache.soft_hash(q, planes, protos, 0.3, 2)
    q[1, 3, 17] = float("nan")
    q[0, 2, 5] = float("inf")
    got = hash_cache.soft_hash(q, planes, protos, 0.3, 2)
    keep = torch.ones(2, 8, dtype=torch.bool, device=DEV)
    keep[1, 3] = keep[0, 2] = False
    assert torch.equal(got[keep], clean[keep]) and got[1, 3].isnan().all()
    # an infinite coordinate saturates every plane it meets
    assert torch.allclose(got[0, 2].double(), exact(q, planes, protos, 0.3)[0, 2], rtol=2 ** -8)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("G", [1, 2, 4])
def test_large_logits_in_some_heads(dtype, G):
    """Logits up to thousands in one head of sixteen: nothing overflows, and the heads beside it have what they have without it."""
    Hq, L, temp = 4 * G, 3, 0.3
    q, planes, protos = inputs(3, Hq, L, G, True)
    q, planes, protos = q.to(dtype), (0.02 * planes).to(dtype), protos.to(dtype) * 16
    planes[1, 4:] *= 1000                                  # (table 1 saturates: logits of up to 16 * 10 / sqrt(128) / 0.3 = 47)
    q[0] *= 0.01
    small = hash_cache.soft_hash(q, planes, protos, temp, 4, out_dtype=torch.float32)
    q2 = q.clone()
    q2[1, 0] *= 100
    got = hash_cache.soft_hash(q2, planes, protos, temp, 4, out_dtype=torch.float32)
    keep = torch.ones(3, Hq, dtype=torch.bool, device=DEV)
    keep[1, 0] = False
    assert torch.equal(got[keep], small[keep])
    want = exact(q2, planes, protos, temp)
    # (logits up to 68 in base 2: sixteen roundings of that size, and where the largest is taken off one more; the projections'
    # 128 products, added up in fp32, are off by 128 * 2^-24 of 128 * 0.02 * 4 in front of a slope of 16 * 10 / sqrt(128) / 0.3)
    bound = 2 ** -23 * (16 + 17 * 68 + 64 * 10 * 47)
    assert ((got.double() - want).abs() <= bound * want + 1e-37).all()
    assert torch.equal(hash_cache.soft_hash(q2, planes, protos, temp, 4, out_dtype=torch.float32, grouped=True)[:, 2, :, :, 0], got[:, 2 * G])
    # far past what an exponential holds: one bucket has it all, and the sums stay finite
    far = hash_cache.soft_hash(q2, planes * 1000, protos * 64, temp, 4, out_dtype=torch.float32)
    assert far.isfinite().all() and torch.allclose(far.sum(-1), torch.ones_like(far[..., 0]), atol=1e-4)


@pytest.mark.parametrize("Hq,Hkv,B", [(8, 8, 3), (28, 4, 5), (6, 3, 7), (16, 4, 1)])
def test_float32_tables_of_every_layout(Hq, Hkv, B):
    """fp32 operands, units that do not fill a workgroup's sixteen heads or cross sequences, padded groups."""
    q, planes, protos = (x.float() for x in inputs(B, Hq, 5, Hq, False))
    parts, width = hash_cache.group_shape(Hq, Hkv)
    G = Hq // Hkv
    want = exact(q, planes, protos, 0.3)
    flat = hash_cache.soft_hash(q, planes, protos, 0.3, Hkv)
    assert ((flat.double() - want).abs() <= 2 ** -23 * (16 + 16 * 0.9 * 4 / 0.3) * want).all()
    got = hash_cache.soft_hash(q, planes, protos, 0.3, Hkv, grouped=True)
    for h in range(Hq):
        kv, g = h // G, h % G
        assert torch.equal(got[:, kv * parts + g // width, :, :, g % width], flat[:, h])
    for g in range(G, parts * width):
        assert (got.view(B, Hkv, parts, 5, 1024, width)[:, :, g // width, :, :, g % width] == 0).all()


def single(B, Hq, L, seed, positive=False):
    """Planes of one coordinate each, which fp32 projects without an error: t is tanh's alone."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = torch.randn(B, Hq, 128, generator=g, device=DEV).bfloat16()
    planes = torch.zeros(L, 10, 128, device=DEV)
    planes.view(-1, 128)[torch.arange(10 * L, device=DEV), torch.arange(10 * L, device=DEV) * 37 % 128] = 1.0
    return (q.abs() if positive else q), planes.bfloat16()


def assert_close(got, want, largest):
    """(Logits up to `largest` in base 2: sixteen roundings of that size, and an exponential and a normalisation to an ulp or two.)"""
    assert ((got.double() - want).abs() <= 2 ** -23 * (16 + 17 * largest) * want + 1e-37).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes", [(64, 1, 1, 1), (1, 1, 1, 64), (0.01, 64, 1, 16), (4096, 4096, 4096, 4096), (1, 4096, 64, 0.01), (8, 7, 6, 5)])
def test_large_logits_in_some_buckets(dtype, sizes):
    """The four waves' buckets of different sizes: each takes its own largest logit off, or none."""
    q, planes = single(3, 8, 3, 5)
    r, k = torch.arange(1024, device=DEV)[None], torch.arange(10, device=DEV)[:, None]
    protos = (((r >> (9 - k)) & 1) * 2.0 - 1) * torch.tensor(sizes, device=DEV, dtype=torch.float32).repeat_interleave(256)
    protos = protos.to(dtype)
    q[0] *= 0.01                                # (heads of small logits beside them)
    got = hash_cache.soft_hash(q.to(dtype), planes.to(dtype), protos, 0.3, 4, out_dtype=torch.float32)
    t = torch.tanh(torch.einsum("bhd,lkd->bhlk", q.double(), planes.double())) / math.sqrt(128)
    logits = torch.einsum("bhlk,kr->bhlr", t, protos.double()) / 0.3 / math.log(2)
    assert_close(got, torch.softmax(logits * math.log(2), -1), logits.abs().amax().item())
    half = hash_cache.soft_hash(q.to(dtype), planes.to(dtype), protos, 0.3, 4, out_dtype=torch.bfloat16)
    # (bfloat16 has eight significant bits: a rounding is off by up to 2^-8 of its result)
    assert ((half.float() - got).abs() <= 2 ** -8 * got + 1e-37).all()


def test_buckets_that_are_out_of_reach():
    """Logits of minus infinity have no weight, also where they are all of a wave's and the other waves' are far below zero."""
    q, planes = single(2, 4, 2, 6, positive=True)
    protos = torch.full((10, 1024), -100.0, device=DEV) - torch.rand(10, 1024, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    for out in (slice(5, 6), slice(256, 512), slice(0, 900)):
        p = protos.clone()
        p[:, out] = -math.inf
        got = hash_cache.soft_hash(q.float(), planes.float(), p, 0.3, 4)
        finite = torch.ones(1024, dtype=torch.bool, device=DEV)
        finite[out] = False
        assert (got[..., out] == 0).all()
        assert_close(got[..., finite], exact(q, planes, protos[:, finite], 0.3), 10 * 101 / math.sqrt(128) / 0.3 / math.log(2))
    assert hash_cache.soft_hash(q.float(), planes.float(), torch.full_like(protos, -math.inf), 0.3, 4).isnan().all()


def test_large_logits_take_no_second_pass():
    """Small and large logits are worked out once each: the launch takes about as long (made twice, 3.3 to 4.7 times as long)."""
    q, planes, protos = inputs(16, 28, 48, 1, True)

    def best(temperature):
        hash_cache.soft_hash(q, planes, protos, temperature, 4)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(10):
                hash_cache.soft_hash(q, planes, protos, temperature, 4)
        times = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            graph.replay()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    assert best(0.01) < 2 * best(0.3)
