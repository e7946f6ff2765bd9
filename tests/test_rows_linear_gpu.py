"""The matrix-vector products of a decode step at the sizes where their chunks, slots and input forms change."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# A lane adds K / 64 products in pairs, the wave's 64 sums are added in six steps: at most K / 128 + 6 roundings of 2^-24 each
# of the largest partial sum, whose root mean square stays below 2^-24 sqrt(K / 128 + 6) of the result's: 8e-7 at K = 20000.
SUM = 2e-6
# A normed row is rounded to bfloat16 (2^-9 of an element at most) before the product: an output is off by at most 2^-9 sqrt(K)
# times the root of the sum of its squared products, and by 2^-9 of that in root mean square over many.
NORMED = 4e-3


def _rms(got, want, scale=None):
    """Root mean square of the difference over that of `scale`, or of the result."""
    got, want = got.double().cpu(), want.double().cpu()
    return ((got - want).square().mean().sqrt() / (want if scale is None else scale).square().mean().sqrt()).item()


def _spread(h, w):
    """The root of the sum of an output's squared products."""
    return (h.square() @ w.double().square().t()).sqrt()


def _bf(g, *shape):
    return torch.randn(*shape, generator=g, dtype=torch.float32).to(torch.bfloat16)


@pytest.fixture
def dev():
    return torch.device("cuda:0")


# K: below, at and behind a vector of 512 and rows of 1024 that lanes hold; below, at and behind a chunk of 2048; four chunks in flight and more; inputs past the registers on their way to LDS, and
# past LDS.  N: no full workgroup, one row too many for one, two and four rows a wave of the persistent launch.
# Rows that are normed: past a CU's LDS with four at 13640, with three and four at 16384.
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("K,N", [(8, 1), (40, 4097), (2040, 5), (2048, 4099), (2056, 8200), (4096, 1030), (8192, 64), (10248, 33),
                                 (13632, 6), (13640, 6), (14336, 40), (16352, 5), (16384, 24), (16392, 7), (20488, 9), (256, 16390), (64, 40000), (512, 4099), (520, 3), (1024, 8200), (1032, 4090),
                                 (1032, 7), (2048, 1023), (2048, 1028)])
def test_products_of_every_form(dev, rows, K, N):
    from socket_amd import layer_ops
    g = torch.Generator().manual_seed(rows * 1000003 + K * 31 + N)
    x, x2 = _bf(g, rows, 1, K), _bf(g, rows, 1, K)
    w, w2, b, b2 = _bf(g, N, K), _bf(g, N, K), _bf(g, N), _bf(g, N)
    d = dict(device=dev)
    p, p2 = x.double() @ w.double().t(), x2.double() @ w2.double().t()
    assert _rms(layer_ops.linear_f32(x.to(**d), w.to(**d)), p, _spread(x.double(), w)) < SUM
    two = layer_ops.linear_terms([(x.to(**d), w.to(**d), 0.75), (x2.to(**d), w2.to(**d), -1.5)])
    assert _rms(two.a, 0.75 * p - 1.5 * p2) < SUM
    n = 70                                          # (more earlier results than lanes)
    res, past, share = torch.randn(rows, 1, N, generator=g), torch.randn(n + 1, rows, 1, N, generator=g), torch.rand(n + 1, generator=g)
    kept = past.to(**d)
    y, none = layer_ops.linear_residual(x.to(**d), w.to(**d), res.to(**d), b.to(**d), layer_ops.Depth(kept, n, share.to(**d)))
    result = res.double() + p + b.double()
    assert none is None and _rms(kept[n], result) < SUM
    assert _rms(y, share[n] * result + (share[:n].double().view(n, 1, 1, 1) * past[:n].double()).sum(0)) < SUM
    if K > 16384:
        return
    normed = NORMED if K > 8 else 2 ** -9 * K ** 0.5
    s, nw, a, pw = torch.randn(rows, 1, K, generator=g), torch.rand(K, generator=g) + 0.5, torch.randn(rows, 1, K, generator=g), torch.rand(K, generator=g) + 0.5
    for pend in (None, layer_ops.Pending(a.to(**d), 0.5, post_w=pw.to(**d)), layer_ops.Pending(a.to(**d), 2.0),
                 layer_ops.Pending(a.to(torch.bfloat16).to(**d), 0.5)):
        t = s.double()
        if pend is not None:
            z = pend.scale_a * pend.a.double().cpu()
            t = t + (z if pend.post_w is None else z * (z.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * pw.double())
        h = t * (t.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * nw.double()
        got_x, y = layer_ops.norm_linear(s.to(**d), pend, nw.to(**d), 1e-5, w.to(**d), f32_out=True, bias=b.to(**d))
        assert _rms(got_x, t) < 1e-6 and _rms(y, h @ w.double().t() + b.double(), _spread(h, w)) < normed
    _, y = layer_ops.norm_linear(s.to(**d), None, nw.to(**d), 1e-5, (w / K ** 0.5).to(**d), up_weight=(w2 / K ** 0.5).to(**d), act="silu", bias=b.to(**d),
                                 up_bias=b2.to(**d))
    h = s.double() * (s.double().square().mean(-1, keepdim=True) + 1e-5).rsqrt() * nw.double()
    gate, up = h @ (w / K ** 0.5).double().t() + b.double(), h @ (w2 / K ** 0.5).double().t() + b2.double()
    assert _rms(y, gate * torch.sigmoid(gate) * up) < 4 * NORMED
    table, ids = _bf(g, 5, K), torch.tensor([[3], [0], [4], [1]][:rows])
    e = table[ids].double() * 1.25
    got_x, y = layer_ops.norm_linear(None, None, nw.to(**d), 1e-5, w.to(**d), f32_out=True, embed=table.to(**d), ids=ids.to(**d), embed_scale=1.25)
    h = e * (e.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * nw.double()
    assert _rms(got_x, e) < 1e-6 and _rms(y, h @ w.double().t(), _spread(h, w)) < normed


@pytest.mark.parametrize("K", [40, 520, 2056, 41000])      # (the last past what LDS holds of two rows)
def test_an_infinity_stays_in_its_row(dev, K):
    """Lanes past a row's end multiply zeros, not what lies behind the row."""
    from socket_amd import layer_ops
    g = torch.Generator().manual_seed(K)
    x, w = _bf(g, 2, 1, K), _bf(g, 9, K)
    x[1, 0, :] = float("inf")
    got = layer_ops.linear_f32(x.to(dev), w.to(dev)).cpu()
    assert _rms(got[0], x[0].double() @ w.double().t()) < SUM
    assert not torch.isfinite(got[1]).any()
    w[3, K - 1] = float("nan")
    got = layer_ops.linear_f32(x[:1].to(dev), w.to(dev)).cpu()[0, 0]
    assert torch.isnan(got[3]) and torch.isfinite(got[torch.arange(9) != 3]).all()


@pytest.mark.parametrize("K", [40, 2056, 4096])
def test_subnormal_operands_and_results_are_kept(dev, K):
    """One product a row, exact in 32 bits: bfloat16 and 32-bit subnormals go in and come out as they are."""
    from socket_amd import layer_ops
    exponents = [(-130, 100), (100, -130), (-133, 20), (-70, -65), (-60, -80), (-133, -10), (-126, 0), (-140, 0)]
    x, w = torch.zeros(1, 1, K), torch.zeros(len(exponents), K)
    for i, (p, q) in enumerate(exponents):
        at = (i * 37 + 5) % K
        x[0, 0, at], w[i, at] = 1.5 * 2.0 ** p if p > -130 else 2.0 ** p, 2.0 ** q
    x, w = x.to(torch.bfloat16), w.to(torch.bfloat16)
    got = layer_ops.linear_f32(x.to(dev), w.to(dev)).double().cpu()
    want = x.double() @ w.double().t()
    assert (want[0, 0, [0, 1, 2, 3, 6]] != 0).all() and torch.equal(got, want.float().double())
