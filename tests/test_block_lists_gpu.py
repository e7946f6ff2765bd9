"""The block-list launch against the literal pipeline on the host, and the 64-key-tile attention at its edges."""
import pytest
import torch

from oracle import block_sparse_oracle as bso
from socket_amd import block_sparse_flash_attention as bsa

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (columns around the 64 of a lane's bits and a register per lane, the 256 and 1024 of the launch's variants, its last
# column and most picks, one column more, which torch sorts; more picks than columns)
@pytest.mark.parametrize("R,C,K,window,causal,diag", [(1, 1, 1, None, True, True), (5, 5, 9, 2, True, True), (64, 64, 8, 4, True, False),
                                                      (65, 65, 12, None, False, True), (256, 257, 8, 300, True, True),
                                                      (70, 1024, 16, 1, False, False), (1030, 1030, 8, 4, True, True), (90, 31, 5, 3, True, True),
                                                      (20, 4096, 256, 3, False, True), (20, 4097, 8, 3, False, True)])
def test_block_level_lists(R, C, K, window, causal, diag):
    g = torch.Generator().manual_seed(R + K)
    for scores in (torch.rand(2, R, C, generator=g), torch.zeros(2, R, C),
                   torch.rand(2, R, C, generator=g).masked_fill(torch.rand(2, R, C, generator=g) < 0.5, float("-inf"))):
        kw = dict(enforce_causal_blocks=causal, force_include_diagonal=diag, window_blocks=window)
        want = bsa.random_walk_indices_from_block_probs(scores, K, **kw)
        got = bsa.random_walk_indices_from_block_probs(scores.to(DEV), K, **kw)
        assert torch.equal(got.cpu(), want) and torch.equal(want, bso.random_walk_indices_from_block_probs(scores, K, causal, diag, window))
        assert (bsa._lists(scores.to(DEV), K, 1, 1, R, causal, diag, window) is None) == (C > 4096)
        view = torch.zeros(2, R, C + 3, device=DEV)[..., :C]
        view.copy_(scores)
        assert torch.equal(bsa.random_walk_indices_from_block_probs(view, K, **kw).cpu(), want)


@pytest.mark.parametrize("Tq,Tk,bm,bn,K,window", [(130, 130, 64, 64, 2, 1), (300, 200, 64, 32, 6, 3), (129, 700, 32, 64, 4, None)])
def test_token_level_lists(Tq, Tk, bm, bn, K, window):
    probs = torch.rand(2, Tq, Tk, generator=torch.Generator().manual_seed(Tq))
    for causal, diag in ((True, True), (False, True), (True, False)):
        kw = dict(enforce_causal_blocks=causal, force_include_diagonal=diag, window_blocks=window)
        assert torch.equal(bsa.random_walk_indices(probs.to(DEV), bm, bn, K, **kw).cpu(), bsa.random_walk_indices(probs, bm, bn, K, **kw))


def test_what_the_launch_leaves_to_torch():
    scores = torch.rand(1, 40, 40, generator=torch.Generator().manual_seed(1))
    for s in (scores.to(DEV).double(), scores.to(DEV).half()):
        assert bsa._lists(s, 4, 1, 1, 40, True, True, 2) is None
    assert bsa._lists(torch.zeros(1, 1, 5000, device=DEV), 4, 1, 1, 1, False, True, 2) is None
    assert torch.equal(bsa.random_walk_indices_from_block_probs(scores.to(DEV).double(), 4, window_blocks=2).cpu(),
                       bsa.random_walk_indices_from_block_probs(scores.double(), 4, window_blocks=2))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,lens,D,K", [(1, (1, 1), 128, 1), (33, (33, 32), 64, 1), (64, (64, 1), 128, 2), (200, (200, 129), 64, 3),
                                        (961, (961, 400), 128, 7)])
def test_attention_at_the_edges(T, lens, D, K, dt):
    g = torch.Generator().manual_seed(T)
    B, H = 2, 4
    q, k, v = (torch.randn(B, H, T, D, generator=g).to(dt) for _ in range(3))
    n = -(-T // 64)
    blocks = bsa.expand_block_index_to_heads(bsa.random_walk_indices_from_block_probs(torch.rand(B, n, n, generator=g), K, window_blocks=2), H)
    seqlens = torch.tensor(lens, dtype=torch.int32)
    got = bsa.random_walk_sparse_attention(q.to(DEV), k.to(DEV), v.to(DEV), seqlens.to(DEV), blocks.to(DEV)).cpu()
    want = bso.block_sparse_attention(q.double(), k.double(), v.double(), seqlens, blocks)
    for b in range(B):
        assert (got[b, :, lens[b]:] == 0).all()
        a, w = got[b, :, :lens[b]].double(), want[b, :, :lens[b]]
        # (a rounding of the weights, one of the result, each half a unit in the last place, and the fp32 sums)
        assert (a - w).norm() / w.norm() < (2 ** -8 if dt == torch.bfloat16 else 2 ** -11)
