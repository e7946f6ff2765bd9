"""The merge of a latent decode step's partial results: as many splits as a wave has lanes and more, fewer and more than are asked
for ahead, splits that saw no key (whatever lies in their memory), one split, more heads than CUs, and ranks that no group of
lanes fills."""
import types

import pytest
import torch

from socket_amd import layer_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rank,rot,H", [(512, 64, 16), (72, 8, 3), (128, 16, 5), (64, 16, 300)])
@pytest.mark.parametrize("tiles", [1, 2, 8, 9, 31, 33, 63, 64, 65, 128])
@pytest.mark.parametrize("share", [1.0, 0.4])
def test_merge(rank, rot, H, tiles, share, monkeypatch):
    cap = 64 * tiles - 5
    length = max(1, int(cap * share))
    splits = layer_ops.latent_splits(cap, 1, H)
    assert splits == (tiles if H <= 16 else min(tiles, 256 // ((H + 15) // 16)))
    g = torch.Generator(device=DEV).manual_seed(tiles + rank)
    rows = torch.randn(1, cap, rank + rot, generator=g, device=DEV).bfloat16()
    q = (2 * torch.randn(1, 1, H, rank + rot, generator=g, device=DEV)).bfloat16()
    w = (torch.randn(H * 24, rank, generator=g, device=DEV) / rank ** 0.5).bfloat16()
    gate = torch.randn(1, 1, H * 24, generator=g, device=DEV)
    scale = (rank + rot) ** -0.5
    made, empty = [], torch.empty

    def poisoned(*shape, **kw):                 # (what the partial results' memory may hold)
        t = empty(*shape, **kw)
        made.append(t.shape)
        return t.fill_(float("nan")) if t.is_floating_point() else t

    monkeypatch.setattr(torch, "empty", poisoned)
    got = layer_ops.latent_attend(q, types.SimpleNamespace(rows=rows, rank=rank, rot=rot, width=rank + rot), scale, w, 24, gate, pos0=length - 1)
    monkeypatch.undo()
    assert (1, splits, H, (rank + 7) // 8 * 8) in made and (1, splits, H, 2) in made
    keys = rows[0, :length].double()
    p = torch.softmax(q[0, 0].double() @ keys.t() * scale, -1)
    want = ((w.double().view(H, 24, rank) @ (p @ keys[:, :rank])[..., None]).flatten() * torch.sigmoid(gate.double().flatten()))
    # (a rounding to bf16; weights are two bf16 numbers, 2^-16 of each, times rows of size 1 and a value product of size 1)
    assert ((got.flatten().double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -14).all()
