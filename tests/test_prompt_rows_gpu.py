"""The row kernels of a prompt pass against the torch operations they stand for."""
import pytest
import torch
from torch.nn import functional as F

from socket_amd import decode_ops
from socket_amd.model import FeedForward, ModelArgs, RMSNorm, apply_rotary_emb

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,S,Hq,Hkv,D,t0,fdt", [(1, 2, 4, 4, 64, 0, torch.bfloat16), (3, 33, 7, 1, 128, 5, torch.float32),
                                                 (2, 130, 6, 2, 8, 1, torch.bfloat16)])
def test_rope_rows_equals_the_separate_operations(B, S, Hq, Hkv, D, t0, fdt, dt):
    g = torch.Generator(device=DEV).manual_seed(S)
    wide = torch.randn(B, S + 1, (Hq + 2 * Hkv) * D + 64, generator=g, device=DEV).to(dt)
    qkv = wide[:, 1:, 64:]                                             # rows with a stride of their own
    ang = torch.rand(S, D // 2, generator=g, device=DEV) * 6
    freqs = torch.stack([ang.cos(), ang.sin()], -1).to(fdt)
    k_cache, v_cache = (torch.randn(B, Hkv, t0 + S + 3, D, generator=g, device=DEV).to(dt) for _ in range(2))
    want_k, want_v = k_cache.clone(), v_cache.clone()
    q, k, v = qkv.split([Hq * D, Hkv * D, Hkv * D], -1)
    want_q = apply_rotary_emb(q.reshape(B, S, Hq, D), freqs)
    want_k[:, :, t0:t0 + S] = apply_rotary_emb(k.reshape(B, S, Hkv, D), freqs).permute(0, 2, 1, 3)
    want_v[:, :, t0:t0 + S] = v.reshape(B, S, Hkv, D).permute(0, 2, 1, 3)
    assert decode_ops.rope_rows_fits(qkv, freqs, k_cache, v_cache)
    got = decode_ops.rope_rows(qkv, freqs, k_cache, v_cache, t0, Hq, Hkv)
    assert torch.equal(got, want_q) and torch.equal(k_cache, want_k) and torch.equal(v_cache, want_v)
    assert not decode_ops.rope_rows_fits(wide[:, 1:, 1:], freqs, k_cache, v_cache)


@pytest.mark.parametrize("dt,unit", [(torch.bfloat16, 2 ** -8), (torch.float16, 2 ** -11), (torch.float32, 2 ** -22)])
@pytest.mark.parametrize("dim", [8, 100, 4096, 9000])
def test_norm_and_feed_forward_modules(dim, dt, unit):
    """Within two roundings of the type of the float64 result; with gradients the modules stay torch's.  A rounding is
    off by a `unit` of its result, or below the type's normal range (float16: 2^-14) by half the spacing there, 2^-25;
    the first one is scaled by a weight of at most 1.5, and the second adds to it: 2 units and a bit, and 2.5 * 2^-25."""
    bound = lambda want: 2.01 * unit * want.abs() + (2.5 * 2 ** -25 if dt == torch.float16 else 0.0)
    g = torch.Generator(device=DEV).manual_seed(dim)
    norm = RMSNorm(dim).to(DEV, dt)
    norm.weight.data.uniform_(0.5, 1.5, generator=g)
    x = (torch.randn(3, 5, dim, generator=g, device=DEV) * 4).to(dt)
    want = x.double() / (x.double().square().mean(-1, keepdim=True) + norm.eps).sqrt() * norm.weight.double()
    with torch.no_grad():
        assert ((norm(x).double() - want).abs() <= bound(want)).all()
    y = norm(x.clone().requires_grad_())
    y.float().sum().backward()
    assert norm.weight.grad is not None and ((y.double() - want).abs() <= bound(want)).all()


def test_feed_forward_module_rounds_as_torch():
    ff = FeedForward(ModelArgs(dim=256, n_head=2, intermediate_size=264)).to(DEV, torch.bfloat16)
    x = torch.randn(2, 37, 256, device=DEV).bfloat16()
    with torch.no_grad():
        want = ff.w2(F.silu(ff.w1(x)) * ff.w3(x))
        got = ff(x)
    # (silu in fp32 by two formulas: now and then the other neighbour in bf16)
    assert (got.float() - want.float()).norm() / want.float().norm() < 2 ** -8
    ff(x).float().sum().backward()
    assert ff.w1.weight.grad is not None
