"""A prompt's residual add inside the norm's launch against the two operations, and the lengths set by the rotary launch."""
import pytest
import torch

from socket_amd import decode_ops
from socket_amd.model import ModelArgs, RMSNorm, Transformer

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dim", [8, 100, 4096, 9000])
def test_add_then_norm(dim, dt):
    g = torch.Generator(device=DEV).manual_seed(dim)
    norm = RMSNorm(dim).to(DEV, dt)
    norm.weight.data.uniform_(0.5, 1.5, generator=g)
    x, r = ((torch.randn(3, 70, dim, generator=g, device=DEV) * 3).to(dt) for _ in range(2))
    with torch.no_grad():
        want = norm(x + r)
        for a, b in ((x, r), (x[:, -1:], r[:, -1:])):              # (whole rows, and rows with a stride of their own)
            h, y = norm.add(a, b)
            assert torch.equal(h, a + b) and torch.equal(y, want[:, -a.shape[1]:])
        seen = []
        hook = norm.register_forward_hook(lambda m, args, out: seen.append(args[0]))
        h, y = norm.add(x, r)                                      # (a hook on the norm sees its input as before)
        hook.remove()
        assert torch.equal(seen[0], x + r) and torch.equal(y, want)
    h, y = norm.add(x.clone().requires_grad_(), r)
    assert h.requires_grad and y.requires_grad


def test_lengths_follow_the_rows():
    lens = torch.full((2,), 99, dtype=torch.int32, device=DEV)
    cache = [torch.zeros(2, 2, 24, 64, device=DEV) for _ in range(2)]
    decode_ops.rope_rows(torch.randn(2, 9, 8 * 64, device=DEV), torch.randn(9, 32, 2, device=DEV), *cache, 7, 4, 2, lens)
    assert lens.tolist() == [16, 16]


@pytest.mark.parametrize("rows", [None, [0, 5, 40]])
def test_chosen_rows_are_those_of_the_whole(rows):
    torch.manual_seed(0)
    cfg = ModelArgs(block_size=128, vocab_size=64, n_layer=2, n_head=4, n_local_heads=2, dim=256, intermediate_size=512)
    model = Transformer(cfg).to(DEV, torch.bfloat16).eval()
    model.setup_caches(2, 64)
    ids, pos = torch.randint(0, 64, (2, 41), device=DEV), torch.arange(41, device=DEV)
    with torch.no_grad():
        whole = model(ids, pos, pos0=0)
        some = model(ids, pos, pos0=0, last_only=rows is None, rows=rows)
    want = whole[:, -1:] if rows is None else whole[:, rows]
    # (one norm and one product of other shapes: bf16's last place at the size of the logits)
    assert (some - want).abs().max() <= 2 ** -7 * want.abs().max()
