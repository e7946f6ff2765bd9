"""build_sparse_list_decode in place (operands in their own types, the list assembled by one launch) against the oracle:
row lengths on and off the 8-token vectors, each workgroup size of the scorer, lists with no base, all base and
positions that are not allowed."""
import pytest
import torch

from oracle import socket_oracle as orc
from socket_amd import sparse

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("qdt,vdt", [(torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16), (torch.float32, torch.float32),
                                     (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("B,H,T,L,P,sink,window,M", [(1, 2, 5, 3, 4, 2, 2, 9), (2, 3, 2056, 12, 6, 4, 64, 100), (1, 2, 4099, 9, 8, 0, 0, 33),
                                                     (1, 40, 30000, 4, 7, 4, 128, 64), (2, 130, 8200, 3, 5, 30, 9000, 50),
                                                      (1, 3, 20000, 3, 5, 3000, 12000, 300), (2, 2, 9000, 3, 5, 0, 4095, 1)])
def test_against_the_oracle(B, H, T, L, P, sink, window, M, qdt, vdt):
    g = torch.Generator().manual_seed(T)
    q = torch.rand(B, H, L, 1 << P, generator=g).to(qdt)
    codes = torch.randint(0, 1 << P, (B, H, L, T), generator=g).to(torch.int16)
    norms = (torch.rand(B, H, T, generator=g) + 0.5).to(vdt)
    allowed = torch.rand(B, H, T, generator=g) < 0.9
    allowed[0, 0, max(1, T // 50):] = False                    # fewer allowed positions than the budget
    want_list, want_len = orc.build_sparse_list_decode(q.float(), codes, norms.float(), allowed, sink, window, M)
    args = [t.to(DEV) for t in (q, codes, norms, allowed)]
    got_list, got_len = sparse.build_sparse_list_decode(*args, sink, window, M)
    assert torch.equal(got_list.cpu(), want_list) and torch.equal(got_len.cpu(), want_len)
    views = [torch.stack([t, t], -1)[..., 0] for t in args]                    # no operand contiguous, codes in 32 bits
    views[1] = views[1].int()
    got_list, got_len = sparse.build_sparse_list_decode(*views, sink, window, M)
    assert torch.equal(got_list.cpu(), want_list) and torch.equal(got_len.cpu(), want_len)


def test_no_heavy_entries_and_errors():
    q = torch.rand(1, 2, 3, 16, device=DEV)
    codes = torch.zeros(1, 2, 3, 20, dtype=torch.int16, device=DEV)
    norms, allowed = torch.ones(1, 2, 20, device=DEV), torch.ones(1, 2, 20, dtype=torch.bool, device=DEV)
    lst, n = sparse.build_sparse_list_decode(q, codes, norms, allowed, 2, 3, 0)
    assert lst[0, 1].tolist() == [0, 1, 17, 18, 19] and (n == 5).all()
    with pytest.raises(RuntimeError):
        sparse.build_sparse_list_decode(q, codes[:, :1], norms, allowed, 2, 3, 4)
    with pytest.raises(RuntimeError):
        sparse.build_sparse_list_decode(q, codes, norms[..., :7], allowed, 2, 3, 4)
