"""Attention over short lists of fp32 rows, a workgroup to a row, against float64; and where that form ends."""
import pytest
import torch

from socket_amd.socket_kernels import sparse_attention_fwd

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D,one_pass", [(128, 256), (64, 512), (32, 1024), (16, 2048)])
@pytest.mark.parametrize("B,H,Hkv", [(1, 5, 1), (2, 32, 8), (3, 6, 3)])
def test_against_float64(D, one_pass, B, H, Hkv):
    g = torch.Generator(device=DEV).manual_seed(D + H)
    T = 700
    q = torch.randn(B, H + 1, D, generator=g, device=DEV)[:, 1:]
    k, v = (torch.randn(B, T, Hkv, D, generator=g, device=DEV).transpose(1, 2) for _ in range(2))
    for width in (1, 15, 33, one_pass - 1, one_pass, one_pass + 1):
        lists = torch.randint(0, T, (B, H, width + 3), generator=g, device=DEV, dtype=torch.int32)[..., :width]
        lists[0, 0, ::3] = -1                                   # (not listed)
        lens = torch.randint(1, width + 1, (B, H), generator=g, device=DEV, dtype=torch.int32)
        lens[-1, -1], lens[0, -1], lens[0, 0] = 0, width + 9, width          # nothing; beyond the list; all
        got = sparse_attention_fwd(q, k, v, lists, lens)
        for b in range(B):
            for h in range(H):
                rows = lists[b, h, :min(int(lens[b, h]), width)].long()
                rows = rows[rows >= 0]
                if rows.numel() == 0:
                    assert got[b, h].isnan().all()
                    continue
                kk, vv = k[b, h * Hkv // H].double()[rows], v[b, h * Hkv // H].double()[rows]
                x = kk @ q[b, h].double() * D ** -0.5
                w = torch.softmax(x, 0)
                # a score is off by (D / 4 + 8) roundings of its absolute sum, a weight by twice that and by its exponential
                # (two hardware units and the argument's own rounding), the sums by 24 roundings of absolute sums
                e = 2 ** -24 * ((D / 4 + 8) * (kk.abs() @ q[b, h].double().abs()) * D ** -0.5).max()
                far = float(x.max() - x.min())
                bound = (2 * e + 2 ** -24 * (far + 64)) * 2 * (w @ vv.abs())
                assert ((got[b, h].double() - w @ vv).abs() <= bound).all(), (width, b, h)
