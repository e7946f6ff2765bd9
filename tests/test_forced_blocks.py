"""The largest number of forced blocks of any row block, as the launch of the block lists is given it: against the masks
that the builders make, over small shapes, and for a shape whose rows nobody would walk through."""
import itertools

import torch

from socket_amd import block_sparse_flash_attention as bsa


def counted(R, C, bm, bn, Tq, causal, diagonal, window):
    """As random_walk_indices masks them."""
    rows, cols = torch.arange(R)[:, None], torch.arange(C)[None]
    valid = cols <= torch.clamp((rows + 1) * bm - 1, max=Tq - 1) // bn if causal else torch.ones(R, C, dtype=torch.bool)
    d = rows * bm // bn
    forced = torch.zeros(R, C, dtype=torch.bool)
    if diagonal:
        forced |= cols == d.clamp(0, C - 1)
    if window > 0:
        forced |= (cols <= d) & (cols >= d - (window - 1))
    forced &= valid
    forced[:, 0] = True
    return int((forced & valid).sum(-1).max())


def test_against_the_masks():
    for (bm, bn), Tq, C in itertools.product([(1, 1), (4, 4), (8, 4), (4, 8), (3, 5), (7, 2)], [1, 5, 16, 23, 40], [1, 2, 3, 6, 11, 30]):
        R = -(-Tq // bm)
        for causal, diagonal, window in itertools.product([True, False], [True, False], [0, 1, 2, 3, 5, 50]):
            shape = (R, C, bm, bn, Tq, causal, diagonal, window)
            assert bsa._most_forced(*shape) == counted(*shape), shape


def test_its_cost_is_that_of_no_loop():
    n = 1 << 40
    assert bsa._most_forced(n, n, 64, 64, n * 64, True, True, 4) == 5
