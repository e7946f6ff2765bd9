"""Rows of which fewer positions are allowed than are asked for: masked positions, thousands of them, are among the entries
that the selection orders, and become -1."""
import pytest
import torch

from socket_amd import sparse

pytestmark = pytest.mark.gpu


def _operands(dev, B, H, T, seed, wide):
    g = torch.Generator(device=dev).manual_seed(seed)
    L, R = 4, 64
    q = torch.rand(B, H, L, R, generator=g, device=dev)
    codes = torch.randint(0, R, (B, H, L, T), generator=g, device=dev).to(torch.int16)
    norms = torch.rand(B, H, T, generator=g, device=dev) + 0.1
    if wide:      # (scores over some thirty powers of two)
        norms = torch.exp(5 * torch.randn(B, H, T, generator=g, device=dev))
    return q, codes, norms, g


def _allowed(where, B, H, T, n, g, dev):
    at = torch.arange(T, device=dev)
    if where == "front":
        keep = at < n
    elif where == "end":
        keep = at >= T - n
    else:
        return torch.rand(B, H, T, generator=g, device=dev).argsort(-1) < n
    return keep.expand(B, H, T).contiguous()


def _same(q, codes, norms, allowed, sink, window, M):
    got, got_len = sparse.build_sparse_list_decode(q, codes, norms, allowed, sink, window, M)
    want, want_len = sparse._build_with_torch(q, codes, norms, allowed, sink, window, M)
    assert torch.equal(got, want) and torch.equal(got_len, want_len)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("where", ["front", "end", "scattered"])
# Short by 1048, 724, 924 and 600 allowed positions, of which all but a last run of some 512 are placed by bin; by 290, all
# in that run; by more than the placement by bin takes; nothing, one and all but one allowed.
@pytest.mark.parametrize("T,n,M", [(8192, 1000, 2048), (4096, 300, 1024), (4096, 100, 1024), (8192, 100, 700), (8192, 410, 700),
                                   (8192, 1000, 4096), (2049, 0, 2048), (2500, 1, 1), (8192, 8191, 8192)])
def test_fewer_allowed_than_asked_for(dev, T, n, M, where, wide):
    q, codes, norms, g = _operands(dev, 2, 4, T, T + n + M, wide)
    _same(q, codes, norms, _allowed(where, 2, 4, T, n, g, dev), 4, 64, M)


@pytest.mark.parametrize("T,n,M", [(8192, 1000, 2048), (4096, 300, 1024), (8192, 100, 700)])
def test_more_rows_than_cus(dev, T, n, M):
    """The half workgroups, some of whose rows have everything allowed and some nothing."""
    H = 16
    B = torch.cuda.get_device_properties(dev).multi_processor_count // H + 1
    q, codes, norms, g = _operands(dev, B, H, T, T + M, False)
    allowed = _allowed("scattered", B, H, T, n, g, dev)
    allowed[1], allowed[2] = True, False
    _same(q, codes, norms, allowed, 4, 64, M)


@pytest.mark.parametrize("seed", range(6))
def test_allowed_by_chance(dev, seed):
    q, codes, norms, g = _operands(dev, 1, 8, 8192, seed, seed % 2 == 1)
    allowed = torch.rand(1, 8, 8192, generator=g, device=dev) < 0.05
    allowed[:, 0, 4096:] = False
    _same(q, codes, norms, allowed, 0, 0, 700)
