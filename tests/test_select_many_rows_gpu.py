"""Selection over more rows than the chip has CUs, whose workgroups are half as wide and keep the pool over their other
LDS: whole numbers against a stable sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scores(kind, rows, T, g, dev):
    s = torch.exp(1.5 * torch.randn(1, rows, T, generator=g, device=dev))
    if kind == "ties":
        s = (s * 4).round() / 4                       # few values, each many times over
    elif kind == "one_value":
        s.fill_(0.25)                                 # no threshold separates anything: from scratch, lowest indices
    elif kind == "misled":
        s[:, :, T // 2:T // 2 + 40] += 1000.0         # a cluster that the sample may miss or hit
        s[:, ::3, :] = torch.linspace(0, 1, T, device=dev)
    elif kind == "extremes":
        s[:, :, ::7] = float("-inf")
        s[:, :, 5] = float("inf")
        s[:, :, 9] = float("nan")
    return s


@pytest.mark.parametrize("extra", [1, 300])
@pytest.mark.parametrize("T,M", [(37, 5), (4096, 300), (8192, 2048), (8193, 1), (8200, 2048), (9001, 129), (20003, 2048), (20000, 2049), (33333, 700)])
@pytest.mark.parametrize("kind", ["plain", "ties", "one_value", "misled", "extremes"])
def test_more_rows_than_cus(dev, kind, T, M, extra):
    from socket_amd import sparse
    rows = torch.cuda.get_device_properties(dev).multi_processor_count + extra
    g = torch.Generator(dev).manual_seed(T + M)
    s = _scores(kind, rows, T, g, dev)
    got, _ = sparse.select_list(s, 4, 32, M)
    want = torch.sort(s, dim=-1, descending=True, stable=True)[1][..., :M].to(torch.int32)
    assert torch.equal(got[..., 36:], want)


@pytest.mark.parametrize("T", [8195, 12001])
def test_more_rows_than_cus_masked_and_ragged(dev, T):
    from socket_amd import sparse
    H = 16
    B = torch.cuda.get_device_properties(dev).multi_processor_count // H + 2
    g = torch.Generator(dev).manual_seed(T)
    s = torch.exp(1.5 * torch.randn(B, H, T, generator=g, device=dev))
    lens = torch.randint(8193, T + 1, (B,), generator=g, device=dev).to(torch.int32)
    lens[0], lens[1] = 40, T                          # (a row shorter than its budget)
    budgets = torch.randint(1, 300, (B,), generator=g, device=dev).to(torch.int32)
    got, n = sparse.select_list(s, 4, 32, 300, lens=lens, budgets=budgets)
    for b in range(B):
        m = min(int(budgets[b]), int(lens[b]))
        want = torch.sort(s[b, :, :int(lens[b])], dim=-1, descending=True, stable=True)[1][..., :m].to(torch.int32)
        assert torch.equal(got[b, :, 36:36 + m], want) and int(n[b, 0]) == 36 + m
    codes = torch.randint(0, 1 << 8, (B, H, 6, T), generator=g, device=dev).to(torch.int16)
    probs = torch.rand(B, H, 6, 256, generator=g, device=dev)
    norms = torch.rand(B, H, T, generator=g, device=dev).half()
    allowed = (torch.arange(T, device=dev)[None, None, :] < lens[:, None, None]).expand(B, H, T).contiguous()
    lst, _ = sparse.build_sparse_list_decode(probs, codes, norms, allowed, 4, 32, 200)
    few, _ = sparse.build_sparse_list_decode(probs[:2], codes[:2], norms[:2], allowed[:2].contiguous(), 4, 32, 200)
    assert torch.equal(lst[:2], few)                  # (two sequences are fewer rows than CUs)
