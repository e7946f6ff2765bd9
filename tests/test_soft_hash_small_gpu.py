"""The soft hash of few buckets (a wave to a head) against float64, in every layout."""
import pytest
import torch

from socket_amd import hash_cache

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,D,L,K,R", [(1, 32, 8, 128, 32, 8, 256), (2, 14, 2, 256, 3, 16, 252), (3, 6, 3, 36, 5, 9, 8),
                                              (1, 8, 1, 4, 2, 1, 4), (2, 5, 5, 64, 4, 7, 128)])
def test_against_float64(B, Hq, Hkv, D, L, K, R, dtype):
    g = torch.Generator().manual_seed(R + D)
    q, planes, protos = (torch.randn(*s, generator=g).to(dtype).cuda() for s in ((B, Hq, D), (L, K, D), (K, R)))
    temp = 0.3
    scale = 1 / (D ** 0.5 * temp)
    qd, pd, sd = q.double(), planes.double(), protos.double()
    z = torch.einsum("bhd,lkd->bhlk", qd, pd)
    t = torch.tanh(z) * scale
    logits = t @ sd
    want = torch.softmax(logits, -1)
    # a logit is off by the projections' error (at most D + 2 roundings of the absolute sum) through tanh's slope of at most 1,
    # by tanh and its scaling (8 units of t) and by its own K sums; a probability by twice that, its exponential's argument
    # and value (its distance from the maximum and 4 units), and the sum and product (R / 64 + 8 additions)
    dz = (D + 2) * U * torch.einsum("bhd,lkd->bhlk", qd.abs(), pd.abs())
    e = (scale * dz + 8 * U * t.abs()) @ sd.abs() + K * U * (t.abs() @ sd.abs())
    e = e.amax(-1, keepdim=True)
    far = logits.amax(-1, keepdim=True) - logits
    bound = (2 * e + U * (far + R / 64 + 16)) * 1.01
    plain = hash_cache.soft_hash(q, planes, protos, temp, Hkv, out_dtype=torch.float32)
    assert ((plain.double() - want).abs() <= bound * want + 2.0 ** -140).all()
    half = hash_cache.soft_hash(q, planes, protos, temp, Hkv, out_dtype=torch.bfloat16)
    assert torch.equal(half, plain.to(torch.bfloat16))
    for out, std in ((torch.float32, plain), (torch.bfloat16, half)):
        grouped = hash_cache.soft_hash(q, planes, protos, temp, Hkv, out_dtype=out, grouped=True)
        assert torch.equal(grouped, hash_cache.group_q_probs(std, Hkv))
    wide = torch.randn(B, Hq, D + 1, generator=g).to(dtype).cuda()[..., :D]         # (rows off a multiple of four elements)
    wide.copy_(q)
    assert ((hash_cache.soft_hash(wide, planes, protos, temp, Hkv, out_dtype=torch.float32).double() - want).abs()
            <= bound * want + 2.0 ** -140).all()
