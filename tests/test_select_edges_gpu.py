"""Selection at the edges of its loads and batches: rows of any length and pitch, the last of them at the end of its
allocation, against a stable sort (NaN first, equal scores by index)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2, 3, 5, 63, 4093, 4097, 8190, 8191, 8193, 8194, 16383, 16385, 32771, 65537])
@pytest.mark.parametrize("kind", ["plain", "ties", "extremes"])
def test_lengths(dev, T, kind):
    from socket_amd import sparse
    g = torch.Generator(dev).manual_seed(T)
    s = torch.exp(1.5 * torch.randn(1, 5, T, generator=g, device=dev))
    if kind == "ties":
        s = (s * 4).round() / 4
    elif kind == "extremes":
        s[:, :, ::7] = float("-inf")
        s[:, ::2, T // 2:T // 2 + 3] = float("nan")
        s[:, 1, T - 1] = float("inf")
    for M in (1, min(T, 129), min(T, 2048)):
        got, n = sparse.select_list(s, 0, 0, M, write_base=False)
        want = torch.sort(s, dim=-1, descending=True, stable=True)[1][..., :M].to(torch.int32)
        assert torch.equal(got, want) and bool((n == M).all()), M
