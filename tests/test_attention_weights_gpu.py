"""What the attention kernels' softmax weights keep: the largest weight of a row is exact, and a row's result depends on
that row alone."""
import math

import pytest
import torch

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
