"""Selection and attention of short rows in one launch against the two launches' list and float64, and where it ends."""
import pytest
import torch

from socket_amd import hash_cache
from socket_amd.sparse import select_attend, select_list

pytestmark = pytest.mark.gpu


def _operands(dev, B, H, Hkv, T, D, dtype, seed):
    g = torch.Generator(dev).manual_seed(seed)
    scores = torch.exp(1.5 * torch.randn(B, H, T + 3, generator=g, device=dev))[..., :T]       # (odd pitches among them)
    scores = (scores * 16).round() / 16 if seed % 2 else scores                                 # (ties)
    q = torch.randn(B, H + 1, D, generator=g, device=dev).to(dtype)[:, 1:]
    k, v = (torch.randn(B, T + 8, Hkv, D, generator=g, device=dev).to(dtype).transpose(1, 2) for _ in range(2))
    return scores, q, k, v


def _sorted_list(scores, sink, window, M):
    """Sink, window and the M largest (NaN first, equal scores by index) of full rows, without the library."""
    B, H, T = scores.shape
    base = torch.tensor([i for i in range(T) if i < sink or i >= T - window], dtype=torch.int32, device=scores.device)
    best = torch.sort(scores, dim=-1, descending=True, stable=True)[1][..., :M].to(torch.int32)
    lists = torch.cat([base.expand(B, H, -1), best], -1)
    return lists, torch.full((B, H), lists.shape[-1], dtype=torch.int32, device=scores.device)


def _check(got, scores, q, k, v, sink, window, M, lens=None, budgets=None, listed=None):
    lists, n = listed or select_list(scores, sink, window, M, lens=lens, budgets=budgets)
    B, H, D = q.shape
    G = H // k.shape[1]
    unit = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[q.dtype]
    for b in range(B):
        for h in range(H):
            rows = lists[b, h, :int(n[b, h])].long()
            rows = rows[rows >= 0]
            if rows.numel() == 0:
                assert got[b, h].isnan().all()
                continue
            kk, vv = k[b, h // G].double()[rows], v[b, h // G].double()[rows]
            x = kk @ q[b, h].double() * D ** -0.5
            w = torch.softmax(x, 0)
            # as in the test of short lists (a score's sum, the exponentials, sums over lanes and waves), and the result's
            # rounding to its type
            e = 2 ** -24 * ((D / 4 + 8) * (kk.abs() @ q[b, h].double().abs()) * D ** -0.5).max()
            far = float(x.max() - x.min())
            want = w @ vv
            bound = (2 * e + 2 ** -24 * (far + 64)) * 2 * (w @ vv.abs()) * (1 + unit) + unit * want.abs() + (2.0 ** -25 if unit else 0)
            assert ((got[b, h].double() - want).abs() <= bound).all(), (b, h)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,M,window,D", [(1, 1, 1, 128), (5, 3, 9, 128), (300, 150, 20, 64), (2000, 0, 30, 128), (4096, 128, 64, 128),
                                          (8191, 100, 0, 64), (8192, 200, 52, 128)])
def test_against_float64(dev, dtype, T, M, window, D):
    ops = _operands(dev, 2, 6, 3, T, D, dtype, T + M)
    got = select_attend(*ops, 4, window, M)
    assert got is not None
    _check(got, *ops, 4, window, M)


# Rows whose m-th bin or bins of winners are full: more entries than are ranked or kept at once, a second pass over them, the
# sort in place of counting.
HARD = {
    "equal": lambda s: s * 0 + 1.25,
    "two values": lambda s: (s > 1).float(),
    "three values": lambda s: (s > 0.5).float() + (s > 6).float(),
    "a crowd above": lambda s: torch.where(s > 4, torch.full_like(s, 1e30), s),        # some 1400 winners in one bin
    "two crowds": lambda s: torch.where(s > 25, torch.full_like(s, 1e30), torch.where(s > 12, torch.full_like(s, 9e29), s)),
    "mostly masked": lambda s: torch.where(s > 12, s, torch.full_like(s, float("-inf"))),
    "all masked": lambda s: torch.full_like(s, float("-inf")),
    "extremes": lambda s: torch.where(s > 20, torch.full_like(s, float("inf")), torch.where(s < 0.1, torch.full_like(s, float("nan")), s)),
    "tiny range": lambda s: 1 + (s * 3).floor() * 2.0 ** -23,
    "wide range": lambda s: torch.where(s > 1, s * 1e30, s * 1e-30),
}


@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("T", [511, 4099, 8192])
@pytest.mark.parametrize("kind", HARD)
def test_hard_rows_against_a_stable_sort(dev, kind, T, dtype, D):
    _, q, k, v = _operands(dev, 1, 4, 2, T, D, dtype, T)
    g = torch.Generator(dev).manual_seed(T + 1)
    scores = HARD[kind](torch.exp(1.5 * torch.randn(1, 4, T, generator=g, device=dev)))
    for M in (1, 129, 400, 476):
        got = select_attend(scores, q, k, v, 4, 32, M)
        assert got is not None
        _check(got, scores, q, k, v, 4, 32, M, listed=_sorted_list(scores, 4, 32, M))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [100, 4100, 8192])
def test_a_step_without_details_is_the_step_with_them(dev, T, dtype):
    L, P, B, H, Hkv, D, M = 12, 8, 2, 8, 2, 128, 150
    _, q, k, v = _operands(dev, B, H, Hkv, T, D, dtype, T)
    q, k, v = q.contiguous(), k[:, :, :T].contiguous(), v[:, :, :T].contiguous()
    g = torch.Generator(dev).manual_seed(T)
    words = torch.randint(0, 2 ** 31 - 1, (B, Hkv, hash_cache.words_per_key(L, P), T), generator=g, device=dev, dtype=torch.int32)
    probs = torch.rand(B, H, L, 1 << P, generator=g, device=dev)
    args = (q, probs, k, v, words, torch.rand(B, Hkv, T, generator=g, device=dev).half(), T, P, 4, 32, M)
    lens = torch.tensor([T, T // 3], dtype=torch.int32, device=dev)
    for more in ({}, {"lens": lens}, {"lens": lens, "budgets": torch.tensor([M, 17], dtype=torch.int32, device=dev)}):
        want, scores, lists, n = hash_cache.sparse_decode_step(*args, return_details=True, **more)
        got = hash_cache.sparse_decode_step(*args, **more)
        if "lens" not in more:
            assert torch.equal(lists.sort(-1)[0], _sorted_list(scores, 4, 32, min(M, T))[0].sort(-1)[0])
        _check(want, scores, q, k, v, 4, 32, M, listed=(lists, n))
        _check(got, scores, q, k, v, 4, 32, M, listed=(lists, n))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ragged(dev, dtype):
    ops = _operands(dev, 5, 4, 2, 3001, 128, dtype, 8)
    lens = torch.tensor([0, 1, 3001, 70, 2999], dtype=torch.int32, device=dev)
    budgets = torch.tensor([9, 9, 100, 0, 300], dtype=torch.int32, device=dev)
    got = select_attend(*ops, 4, 32, 120, lens=lens, budgets=budgets)
    _check(got, *ops, 4, 32, 120, lens=lens, budgets=budgets)


@pytest.mark.parametrize("dtype,D,most", [(torch.float32, 128, 256), (torch.float32, 64, 512), (torch.bfloat16, 128, 512),
                                          (torch.float16, 64, 512)])
def test_where_it_ends(dev, dtype, D, most):
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    for T, H, M, taken in ((8192, 2, most - 36, True), (8192, 2, most - 35, False), (8193, 2, 100, False), (700, cus, 100, True),
                           (700, cus + 1, 100, False)):
        ops = _operands(dev, 1, H, 1, T, D, dtype, 4)
        got = select_attend(*ops, 4, 32, M)
        assert (got is not None) == taken, (T, H, M)
        if taken and H < cus:
            _check(got, *ops, 4, 32, M)
    ops = _operands(dev, 1, 2, 1, 64, 32, dtype, 4)             # (heads of 32 dims: two launches)
    assert select_attend(*ops, 4, 8, 8) is None


def test_misaligned_rows_are_refused(dev):
    scores, q, k, v = _operands(dev, 1, 2, 1, 100, 64, torch.float32, 2)
    with pytest.raises(RuntimeError):
        select_attend(scores, torch.cat([q, q], -1)[..., 1:65], k, v, 4, 8, 8)
