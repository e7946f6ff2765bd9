"""The decode step's one-launch head for fp32 models and for few buckets (bf16 with ten planes: test_model_gpu.py)."""
import pytest
import torch

from socket_amd import decode_ops, hash_cache
from socket_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,Hq,Hkv,L,K,R,grouped,ftype", [
    (torch.float32, 32, 8, 32, 8, 256, True, torch.bfloat16),
    (torch.float32, 28, 4, 5, 8, 256, True, torch.float32),       # two parts of a group, a word that is not full
    (torch.float32, 6, 6, 3, 3, 8, False, torch.float32),         # two lanes with buckets
    (torch.bfloat16, 28, 4, 32, 8, 256, True, torch.bfloat16),
    (torch.bfloat16, 16, 8, 7, 12, 128, False, torch.float32),    # more than eight planes
    (torch.float32, 32, 8, 60, 10, 1024, True, torch.bfloat16),   # the fp32 matrix products: units of four heads,
    (torch.float32, 28, 4, 33, 10, 1024, True, torch.float32),    # ... with filled-up units
    (torch.float32, 16, 8, 7, 10, 1024, True, torch.float32),     # ... of two
    (torch.float32, 5, 5, 2, 10, 1024, False, torch.bfloat16),    # ... and of one
])
def test_prologue_of_other_types_equals_the_three_launches(dt, Hq, Hkv, L, K, R, grouped, ftype):
    """Bit for bit what rope_append, hash_keys and soft_hash leave, also for positions outside the cache or the rotary table;
    the table as near float64 as fp32 sums are."""
    dev, B, D, Tcap, n_pos = "cuda", 3, 128, 72, 70
    g = torch.Generator().manual_seed(Hq + L)
    qkv = (torch.randn(B, 1, (Hq + 2 * Hkv) * D, generator=g) * 2).to(dt).to(dev)
    table = M.precompute_freqs_cis(n_pos, D, 10000).to(ftype).to(dev)
    planes = (torch.randn(L, K, D, generator=g) * 0.3).to(dt).to(dev)
    protos_T = torch.randn(K, R, generator=g).to(dt).to(dev)
    words, NW = hash_cache.permute_planes(planes), hash_cache.words_per_key(L, K)
    assert hash_cache.decode_prologue_fits(qkv, D, K, R, Hq, Hkv)

    def fresh():
        gg = torch.Generator().manual_seed(5)
        return ([torch.randn(B, Hkv, Tcap, D, generator=gg).to(dt).to(dev) for _ in range(2)] +
                [torch.randint(0, 2 ** 31 - 1, (B, Hkv, NW, Tcap), generator=gg, dtype=torch.int32).to(dev),
                 torch.rand(B, Hkv, Tcap, generator=gg).half().to(dev), torch.tensor([3, 10, 1], dtype=torch.int32, device=dev)])

    for ip in ([17], [0, 69, 71], [72, -1, 5]):
        ip, a, b = torch.tensor(ip, device=dev), fresh(), fresh()
        q_a, kn, vn = decode_ops.rope_append(qkv, table, ip, a[0], a[1], a[4], Hq, Hkv, return_new=True)
        hash_cache.hash_keys_into(kn, vn, words, a[2], a[3], L, K, pos_b=ip.to(torch.int32).expand(B).contiguous(), layout="bshd")
        t_a = hash_cache.soft_hash(q_a, planes, protos_T, 0.7, Hkv, grouped=grouped)
        q_b, t_b = hash_cache.decode_prologue(qkv, table, ip, b[0], b[1], b[4], words, b[2], b[3], planes, protos_T, Hq, Hkv,
                                              temperature=0.7, grouped=grouped)
        assert torch.equal(q_a, q_b) and torch.equal(t_a, t_b)
        for x, y, name in zip(a, b, ("k_cache", "v_cache", "codes", "v_norm", "lens")):
            assert torch.equal(x, y), (name, ip.tolist())
    proj = torch.einsum("bhd,lkd->bhlk", q_b.double(), planes.double())
    scale = 1 / (D ** 0.5 * 0.7)
    want = torch.softmax(torch.tanh(proj) @ protos_T.double() * scale, -1)
    plain = hash_cache.soft_hash(q_b, planes, protos_T, 0.7, Hkv)
    # a sum of n products is off by at most n u sum |products|, tanh carries that on undiminished at most; so the logits are
    # off by that of the projections times the prototypes and (K + 2) u of their own, a ratio of exponentials by twice as much
    u = 2.0 ** -24
    of_proj = D * u * torch.einsum("bhd,lkd->bhlk", q_b.double().abs(), planes.double().abs()) + 4 * u
    of_logit = ((of_proj + (K + 2) * u) @ protos_T.double().abs()).amax(-1, keepdim=True) * scale
    bound = 2 * of_logit + 16 * u + (0 if dt == torch.float32 else 2.0 ** -8)
    assert (((plain.double() - want).abs() / want) <= bound).all()


@pytest.mark.parametrize("moved", ["planes", "protos_T"])
@pytest.mark.parametrize("dt,K,R", [(torch.float32, 8, 256), (torch.float32, 10, 1024), (torch.bfloat16, 4, 16)])
def test_operands_that_start_on_no_boundary(dt, K, R, moved):
    """Views one element into an allocation: such a step is answered by the three launches."""
    dev, B, D, Hq, Hkv, L = "cuda", 2, 128, 8, 4, 6
    cfg = M.ModelArgs(block_size=64, vocab_size=64, n_layer=1, n_head=Hq, n_local_heads=Hkv, dim=Hq * D, intermediate_size=256,
                      head_dim=D, L=L, K=K, R=R)
    steps = []
    for shift in (0, 1):
        torch.manual_seed(1)
        att = M.Attention(cfg).to(device=dev, dtype=dt)
        att.kv_cache = M.KVCache(B, 64, Hkv, D, L=L, R=R, dtype=dt, K=K, device=dev)
        att.sync_planes()
        t = getattr(att, moved)
        whole = torch.empty(t.numel() + shift, dtype=t.dtype, device=dev)
        view = whole[shift:].view(t.shape)
        view.copy_(t)
        setattr(att, moved, view)
        assert (view.data_ptr() % 16 == 0) == (shift == 0)
        qkv = torch.randn(B, 1, (Hq + 2 * Hkv) * D, generator=torch.Generator().manual_seed(3)).to(dt).to(dev)
        freqs = M.precompute_freqs_cis(64, D, 10000).to(torch.float32).to(dev)
        pos = torch.tensor([5], device=dev)
        fused = M._decode_prologue(qkv, freqs, pos, att.kv_cache, att.planes, att.protos_T, Hq, Hkv)
        assert (fused is None) == (shift == 1)
        steps.append(att._run_fused_qkv(qkv, pos, True, M.DecodeStep(freqs, pos.to(torch.int32).expand(B).contiguous())))
    # (every cached token is attended to: the table decides their order alone, and 32-bit sums over 64 of them and 1024
    # columns, or their rounding to bfloat16, are what differs)
    assert torch.isfinite(steps[0]).all()
    assert (steps[0] - steps[1]).float().norm() <= (1e-6 if dt == torch.float32 else 2.0 ** -8) * steps[0].float().norm()
