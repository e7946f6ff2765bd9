"""What the attention kernels' softmax weights keep: the largest weight of a row is exact, a row's result depends on that
row alone, and over a cache the weights have 32 bits."""
import math

import pytest
import torch

from socket_amd import block_sparse_flash_attention as bsa
from socket_amd import layer_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_UNIT = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}      # of results in [1/2, 1)


def few_keys(S, D, dt, scores):
    """Keys [S,D] for queries (1, x, 1, 0 ..) whose scores are those of `scores` (key -> (constant, factor of x)); every
    other key scores -200, a weight of 0 in 32 bits."""
    k = torch.zeros(S, D, device=DEV)
    k[:, 2] = -200.0
    for at, (c, f) in scores.items():
        k[at, 0], k[at, 1], k[at, 2] = c, f, 0.0
    return k.to(dt)


def queries(x, D, dt):
    q = torch.zeros(x.numel(), D, device=DEV)
    q[:, 0], q[:, 1], q[:, 2] = 1.0, x, 1.0
    return q.to(dt)


def late_maximum(dt, n, first, S, D):
    """Two live keys, the later one larger by x / 2 < 5.6 (2^8 in weight): queries, keys, values and the later one's weight."""
    x = torch.linspace(0.25, 11, n, device=DEV).to(dt)
    k = few_keys(S, D, dt, {3: (0.0, 0.0), first: (0.0, 0.5)})
    v = torch.zeros(S, D, device=DEV, dtype=dt)
    v[3, 0] = v[first, 1] = 1.0
    return queries(x.float(), D, dt), k, v, torch.sigmoid(x.double() / 2)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("w16", [True, False])
def test_the_largest_weight_of_a_prompt_row_is_exact(dt, D, w16):
    """It is 1 wherever its key stands, so its value's coordinate is rounded once: half a unit, and 32-bit sums."""
    T, S = 300, 600
    q, k, v, want = late_maximum(dt, T, S - T - 5, S, D)
    got = layer_ops.prompt_attend(q[None, :, None], k[None, :, None], v[None, :, None], S - T, 1.0, weights16=w16)[0, :, 0, 1]
    assert (got.double() - want).abs().max() < 1.01 * HALF_UNIT[dt]


@pytest.mark.parametrize("gain", [3.0, 1e7])
@pytest.mark.parametrize("w16", [True, False])
def test_a_prompt_row_does_not_depend_on_its_neighbours(w16, gain):
    g = torch.Generator(device=DEV).manual_seed(1)
    q = torch.randn(1, 400, 4, 128, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(1, 400, 2, 128, generator=g, device=DEV).bfloat16() for _ in range(2))
    beside = q.clone()
    beside[:, 1::2] *= gain
    beside[:, :, 1::2] *= gain
    a, b = (layer_ops.prompt_attend(x, k, v, 0, 128 ** -0.5, weights16=w16) for x in (q, beside))
    assert torch.equal(a[:, ::2, ::2], b[:, ::2, ::2])


def blocks_of(r):
    """A list per row block: the first, three between, the two before the diagonal, the diagonal."""
    return sorted({0, r // 4, r // 3, r // 2, max(r - 2, 0), max(r - 1, 0), r})


def block_lists(H, R):
    idx = torch.full((1, H, R, 7), R - 1, dtype=torch.int32)      # (padded with a block past the row: nothing visible)
    for r in range(R - 1):
        b = blocks_of(r)
        idx[:, :, r, :len(b)] = torch.tensor(b, dtype=torch.int32)
    idx[:, :, R - 1, :] = torch.arange(R - 7, R, dtype=torch.int32)
    return idx.to(DEV)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
def test_the_largest_weight_of_a_block_sparse_row_is_exact(dt, D):
    """Row block 9 lists blocks 0 and 8 (keys 3 and 512 are live)."""
    T = 640
    q, k, v, want = late_maximum(dt, 64, 512, T, D)
    rows = torch.zeros(T, D, device=DEV, dtype=dt)
    rows[576:] = q
    idx = torch.zeros(1, 1, 10, 2, dtype=torch.int32, device=DEV)
    idx[..., 1] = 8
    # (scores are divided by sqrt(D))
    got = bsa.random_walk_sparse_attention(rows[None, None], (k.float() * 8).to(dt)[None, None], v[None, None],
                                           torch.tensor([T], dtype=torch.int32, device=DEV), idx)[0, 0, 576:, 1]
    want = want if D == 64 else torch.sigmoid(q[:, 1].double() * 4 / D ** 0.5)
    assert (got.double() - want).abs().max() < 1.01 * HALF_UNIT[dt]


@pytest.mark.parametrize("gain", [3.0, 1e7])
@pytest.mark.parametrize("D", [64, 128])
def test_a_block_sparse_row_does_not_depend_on_its_neighbours(D, gain):
    g = torch.Generator(device=DEV).manual_seed(2)
    q, k, v = (torch.randn(1, 2, 700, D, generator=g, device=DEV).bfloat16() for _ in range(3))
    beside = q.clone()
    beside[:, :, 1::2] *= gain
    lens = torch.tensor([700], dtype=torch.int32, device=DEV)
    a, b = (bsa.random_walk_sparse_attention(x, k, v, lens, block_lists(2, 11)) for x in (q, beside))
    assert torch.equal(a[:, :, ::2], b[:, :, ::2])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("counted", [True, False])
def test_weights_over_a_cache_hold_32_bits(D, counted):
    """Row r has in column r the value 1 under a weight p in [1/2, 1) and, under weights of 1, the first two bfloat16 terms of
    -p: what is left is p's last eight bits, at most 2^-18, to the 2^-22 of the exponential's and the sums' 32 bits."""
    x = torch.linspace(0.1, 0.69, D, device=DEV).bfloat16()
    p = torch.exp(-x.double())
    first = p.bfloat16().double()
    second = (p - first).bfloat16().double()
    T, S = D, D + 500
    k = few_keys(S, D, torch.bfloat16, {70: (0.0, 0.0), 150: (0.0, 0.0), 200: (0.0, -1.0)})
    v = torch.zeros(S, D, device=DEV, dtype=torch.bfloat16)
    v[70], v[150], v[200] = -first.bfloat16(), -second.bfloat16(), 1.0
    pos = None if counted else torch.arange(S - T, S, device=DEV)
    got = layer_ops.prompt_attend(queries(x.float(), D, torch.bfloat16)[None, :, None], k[None, :, None], v[None, :, None], S - T,
                                  1.0, pos)[0, :, 0].diagonal().double()
    left = p - first - second
    assert left.abs().max() > 2.0 ** -19
    assert (got * (2 + p) - left).abs().max() < 2.0 ** -21


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_many_small_weights_over_a_cache(dt):
    """4096 weights of about 1.3 x 2^-18 beside one of 1, whose value is 0: small ones keep their bits in fp16 too."""
    S, D = 4097, 64
    c = torch.tensor(math.log(1.3 * 2.0 ** -18)).to(dt)
    k = torch.zeros(S, D, device=DEV, dtype=dt)
    k[1:, 0] = c.to(DEV)
    v = torch.ones(S, D, device=DEV, dtype=dt)
    v[0] = 0
    q = torch.zeros(1, 1, 1, D, device=DEV, dtype=dt)
    q[..., 0] = 1
    got = layer_ops.prompt_attend(q, k[None, :, None], v[None, :, None], S - 1, 1.0).double()
    p = 4096 * math.exp(float(c.double()))
    # (the score in base 2 is rounded to 2^-20 of a unit, which is 2^-20 of the weight)
    assert (got / (p / (1 + p)) - 1).abs().max() < HALF_UNIT[dt] * 2 * 1.01
