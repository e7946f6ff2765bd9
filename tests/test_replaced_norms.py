"""Norms that a caller has put in the decoder's place, or given another forward, are called as they are."""
import pytest
import torch

from socket_amd.model import ModelArgs, Transformer, precompute_freqs_cis


def decoder(device):
    """Without a cache: a prompt by itself."""
    torch.manual_seed(0)
    model = Transformer(ModelArgs(block_size=32, vocab_size=64, n_layer=2, n_head=2, dim=128, intermediate_size=128,
                                  L=4, K=4, R=16)).to(device).eval()
    model.freqs_cis = precompute_freqs_cis(32, 64).to(device)
    model.max_seq_length = 32
    return model


def prompt(model, device):
    ids = torch.arange(12, device=device)[None] % 7
    with torch.no_grad():
        return model(ids, torch.arange(12, device=device), pos0=0)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_replaced_norms(device):
    model = decoder(device)
    want = prompt(model, device)
    for owner, name in [(model, "norm")] + [(b, n) for b in model.layers for n in ("attention_norm", "ffn_norm")]:
        other = torch.nn.RMSNorm(128, eps=model.config.norm_eps).to(device)
        other.load_state_dict(getattr(owner, name).state_dict())
        setattr(owner, name, other)
    assert torch.allclose(prompt(model, device), want, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_a_norm_with_a_forward_of_its_own(device):
    model = decoder(device)
    calls = []
    for b in model.layers:
        b.ffn_norm.forward = lambda x: (calls.append(x.shape), x)[1]
    prompt(model, device)
    assert calls == [(1, 12, 128)] * 2
