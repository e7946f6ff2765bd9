"""The merge of a latent decode step's partial results: as many splits as a wave has lanes and more, fewer and more than are asked
for ahead, splits that saw no key (whatever lies in their memory), one split, and ranks that no group of lanes fills."""
import types

import pytest
import torch

from socket_amd import layer_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rank,rot,H", [(512, 64, 16), (72, 8, 3), (128, 16, 5)])
@pytest.mark.parametrize("tiles", [1, 2, 8, 9, 31, 33, 64, 65, 128])
@pytest.mark.parametrize("share", [1.0, 0.4])
def test_merge(rank, rot, H, tiles, share):
    cap = 64 * tiles - 5
    length = max(1, int(cap * share))
    assert layer_ops.latent_splits(cap, 1, H) == tiles
    g = torch.Generator(device=DEV).manual_seed(tiles + rank)
    rows = torch.randn(1, cap, rank + rot, generator=g, device=DEV).bfloat16()
    q = (2 * torch.randn(1, 1, H, rank + rot, generator=g, device=DEV)).bfloat16()
    w = (torch.randn(H * 24, rank, generator=g, device=DEV) / rank ** 0.5).bfloat16()
    gate = torch.randn(1, 1, H * 24, generator=g, device=DEV)
    scale = (rank + rot) ** -0.5
    rest = torch.full((1 << 24,), float("nan"), device=DEV)
    del rest                                    # (what the partial results' memory may hold)
    got = layer_ops.latent_attend(q, types.SimpleNamespace(rows=rows, rank=rank, rot=rot, width=rank + rot), scale, w, 24, gate, pos0=length - 1)
    keys = rows[0, :length].double()
    p = torch.softmax(q[0, 0].double() @ keys.t() * scale, -1)
    want = ((w.double().view(H, 24, rank) @ (p @ keys[:, :rank])[..., None]).flatten() * torch.sigmoid(gate.double().flatten()))
    # (a rounding to bf16; weights are two bf16 numbers, 2^-16 of each, times rows of size 1 and a value product of size 1)
    assert ((got.flatten().double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -14).all()
