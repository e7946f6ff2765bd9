"""What the launch of selection and attention together refuses or leaves to the two launches, as these had it."""
import ctypes

import pytest
import torch

from socket_amd import _lib, hash_cache, sparse


def test_the_entry_takes_no_larger_budget_than_the_selection():
    nul, one = ctypes.c_void_p(0), ctypes.c_void_p(16)      # (never dereferenced: the budget is looked at first)

    def call(M):
        return _lib.lib().socket_select_attend(one, 64, nul, nul, 64, M, 4, 8, 76, one, one, one, _lib.SOCKET_F32, 256, 128, 8192, 8192,
                                               128, 8192, 8192, 128, one, 256, 128, 1, 2, 1, 128, 64, nul)

    assert call(_lib.SOCKET_TOPK_MAX_M + 1) == _lib.SOCKET_ERR_UNSUPPORTED
    assert _lib.lib().socket_select_list(one, 64, nul, nul, nul, 0, 1, 2, 64, _lib.SOCKET_TOPK_MAX_M + 1, 4, 8, 1, one, 76, 76, nul, nul,
                                         0, nul) == _lib.SOCKET_ERR_UNSUPPORTED
    z = torch.zeros(1, 2, 64)
    with pytest.raises(RuntimeError, match="exceeds the supported maximum"):
        sparse.select_attend(z, torch.zeros(1, 2, 128), torch.zeros(1, 1, 64, 128), torch.zeros(1, 1, 64, 128), 4, 8,
                             _lib.SOCKET_TOPK_MAX_M + 1)


def test_operands_that_do_not_agree_with_the_scores_are_not_read():
    B, H, T, D = 2, 4, 50, 64
    s, q, k = torch.zeros(B, H, T), torch.zeros(B, H, D), torch.zeros(B, 2, T, D)
    n = torch.zeros(B, dtype=torch.int32)
    agree = sparse._rows_agree
    assert agree(s, q, k, k, None, None) and agree(s, q, k, k, n, n)
    assert agree(s, q, torch.zeros(B + 1, 2, T, D), torch.zeros(B + 1, 2, T, D), n, None)      # (a cache of more sequences)
    assert not agree(s, q[:1], k, k, n, n)
    assert not agree(s, q[:, :2], k, k, n, n)
    assert not agree(s, q, k[:1], k[:1], n, n)
    assert not agree(s, q, k, k[:1], n, n)
    assert not agree(s, q, k, k[:, :, 1:], n, n)
    assert not agree(s, q, k, k, n.long(), n)
    assert not agree(s, q, k, k, n, n.long())
    assert not agree(s, q, k, k, n[:1], n)
    assert not agree(s, q, k, k, n, n[:1].expand(B))
    assert not agree(s, q, k, k, n, n.to("meta"))
    # such a call goes on to the two launches: nothing is handed to the library here
    assert sparse.select_attend(s, q[:1], k, k, 1, 1, 4) is None


@pytest.mark.gpu
def test_a_step_refuses_a_large_budget_at_any_length(dev):
    L, P, D = 8, 8, 128
    for T in (64, 9000):
        k = torch.randn(1, 2, T, D, device=dev)
        codes = torch.zeros(1, 2, hash_cache.words_per_key(L, P), T, dtype=torch.int32, device=dev)
        with pytest.raises(RuntimeError, match="exceeds the supported maximum"):
            hash_cache.sparse_decode_step(torch.randn(1, 4, D, device=dev), torch.rand(1, 4, L, 1 << P, device=dev), k, k, codes,
                                          torch.rand(1, 2, T, device=dev).half(), T, P, 4, 16, _lib.SOCKET_TOPK_MAX_M + 1)
