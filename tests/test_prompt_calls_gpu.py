"""Prompt passes in the forms that callers may give them."""
import pytest
import torch

from socket_amd import layer_ops
from socket_amd.model import ModelArgs, Transformer

pytestmark = pytest.mark.gpu


def decoder(dtype=torch.bfloat16, batch=1):
    torch.manual_seed(1)
    model = Transformer(ModelArgs(block_size=64, vocab_size=96, n_layer=2, n_head=2, dim=128, intermediate_size=128,
                                  L=4, K=4, R=16)).to("cuda", dtype).eval()
    with torch.device("cuda"):
        model.setup_caches(batch, 64)
    return model


@torch.no_grad()
def test_a_portion_with_positions_of_any_stride():
    model = decoder()
    ids = torch.randint(0, 96, (1, 30), device="cuda")
    pos = torch.arange(30, device="cuda")
    column = torch.stack([pos, pos + 7], 1)[:, 0]
    want = [model(ids[:, :11], pos[:11], pos0=0), model(ids[:, 11:], pos[11:], pos0=11)]
    got = [model(ids[:, :11], column[:11], pos0=0), model(ids[:, 11:], column[11:], pos0=11)]
    assert not column.is_contiguous() and all(torch.equal(a, b) for a, b in zip(got, want))


def test_empty_tensors():
    q = torch.zeros(0, 5, 2, 64, device="cuda", dtype=torch.bfloat16)
    assert not layer_ops.prompt_attend_fits(q, q, q)


def test_scales_the_kernel_does_not_take():
    """Zero (a mean over the keys) and below are left to torch's attention."""
    q = torch.randn(1, 9, 2, 64, device="cuda").bfloat16()
    assert layer_ops.prompt_attend_fits(q, q, q, 0.1)
    for scale in (0.0, -0.1, float("nan")):
        assert not layer_ops.prompt_attend_fits(q, q, q, scale)


@torch.no_grad()
def test_weights_keep_32_bits_where_flash_kernels_are_switched_off():
    """As torch's attention then does.  Values of +1 and -1 under weights 1 and p leave (1 - p) / (1 + p), of which weights
    in bfloat16 leave a multiple of 2^-9."""
    att = decoder().layers[0].attention
    q, k, v = (torch.zeros(1, 2, 2, 64, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    q[..., 0], k[:, 0, :, 0] = 1.0, -0.01171875
    v[:, 0], v[:, 1] = -1.0, 1.0
    want = torch.tanh(torch.tensor(0.01171875 / 8 / 2, dtype=torch.float64)).item()
    pos = torch.arange(2, device="cuda")
    with torch.nn.attention.sdpa_kernel(torch.nn.attention.SDPBackend.MATH):
        exact = att._prefill_attention(q, k, v, pos, 0)[0, 1, 0, 0].item()
    flash = att._prefill_attention(q, k, v, pos, 0)[0, 1, 0, 0].item()
    assert abs(exact / want - 1) < 2.0 ** -8 and abs(flash / want - 1) > 2.0 ** -3
