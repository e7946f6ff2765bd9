"""What a short decode step, whose selection and attention are one launch, leaves as the two launches left it: the one-launch
attention's scratch array is looked up for a longer step recorded later, and a warm-up loads what that step will run."""
import pytest
import torch

from socket_amd import generate, hash_cache
from socket_amd.model import ModelArgs, Transformer

pytestmark = pytest.mark.gpu


def _operands(dev, B, T):
    L, P, D, Hq, Hkv = 8, 8, 64, 32, 8
    g = torch.Generator(dev).manual_seed(T)
    q = torch.randn(B, Hq, D, generator=g, device=dev)
    probs = torch.rand(B, Hq, L, 1 << P, generator=g, device=dev)
    k, v = (torch.randn(B, Hkv, T, D, generator=g, device=dev) for _ in range(2))
    words = torch.randint(0, 2 ** 31 - 1, (B, Hkv, hash_cache.words_per_key(L, P), T), generator=g, device=dev, dtype=torch.int32)
    return q, probs, k, v, words, torch.rand(B, Hkv, T, generator=g, device=dev).half(), T, P, 4, 16, 64


def _step(*operands, **more):
    return hash_cache.sparse_decode_step(*operands, **more)


@pytest.mark.parametrize("T", [512, 9000])
@pytest.mark.parametrize("rows", [32, 128])
def test_an_eager_step_looks_the_scratch_array_up(dev, monkeypatch, rows, T):
    monkeypatch.setattr(hash_cache, "_STATIC_READY", set())
    ops = _operands(dev, rows // 32, T)
    assert torch.isfinite(_step(*ops, one_launch=False)).all()
    assert hash_cache._STATIC_READY == set()
    _step(*ops)
    assert hash_cache._STATIC_READY == {dev.index}


def test_a_long_step_recorded_after_a_short_one_is_one_launch(dev, monkeypatch):
    monkeypatch.setattr(hash_cache, "_STATIC_READY", set())
    _step(*_operands(dev, 4, 512))
    taken = []
    static = hash_cache.sparse_attention_fwd_static
    monkeypatch.setattr(hash_cache, "sparse_attention_fwd_static", lambda *a: taken.append(1) or static(*a))
    ops = _operands(dev, 4, 9000)
    want = _step(*ops, one_launch=False)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = _step(*ops)
    assert taken == [1]
    for _ in range(3):
        g.replay()
        assert torch.equal(got, want)


def test_warm_up_runs_both_forms(dev, monkeypatch):
    args = ModelArgs(block_size=512, vocab_size=64, n_layer=1, n_head=4, dim=256, n_local_heads=2, L=8, R=256, K=8, heavy_const=64,
                     sink_size=4, window_size=16)
    model = Transformer(args).to(dev, torch.bfloat16)
    ran = set()
    for name in ("select_attend", "select_list", "sparse_attention_fwd"):
        fn = getattr(hash_cache, name)

        def seen(*a, _fn=fn, _name=name, **kw):
            out = _fn(*a, **kw)
            if out is not None:
                ran.add(_name)
            return out
        monkeypatch.setattr(hash_cache, name, seen)
    generate.warmup_sparse_decode(model, dev, T=300)
    assert ran == {"select_attend", "select_list", "sparse_attention_fwd"}
