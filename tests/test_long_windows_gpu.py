"""Lists whose window is long: written by several workgroups, in a launch of their own."""
import pytest
import torch

from socket_amd import sparse

pytestmark = pytest.mark.gpu


class _Watched:
    """The library, with the names of the entry points that are called noted down."""

    def __init__(self, lib):
        self._lib, self.called = lib, []

    def __getattr__(self, name):
        f = getattr(self._lib, name)

        def call(*args):
            self.called.append(name)
            return f(*args)
        return call


@pytest.mark.parametrize("B,H,T,sink,window,kept", [
    (1, 4, 32768, 4, sparse._LONG_BASE - 4, 1.0),      # the longest that the selection's launch writes
    (1, 4, 32768, 4, sparse._LONG_BASE - 3, 0.6),      # ... and one more
    (1, 3, 30001, 7, 30001, 0.5),                      # the whole row, the sink in it; no multiple of a workgroup's entries
    (2, 2, 40000, 30000, 5000, 0.9),                   # a long sink
    (1, 2, 100000, 0, 100000, 0.3),
    (1, 300, 25000, 0, 24900, 0.7),                    # more rows than CUs
])
def test_long_windows(dev, monkeypatch, B, H, T, sink, window, kept):
    L, R, M = 3, 32, 129
    g = torch.Generator(device=dev).manual_seed(T + window)
    q = torch.rand(B, H, L, R, generator=g, device=dev)
    codes = torch.randint(0, R, (B, H, L, T), generator=g, device=dev).to(torch.int16)
    norms = (torch.rand(B, H, T, generator=g, device=dev) + 0.1).half()
    allowed = torch.rand(B, H, T, generator=g, device=dev) < kept
    allowed[:, 0, :T // 2] = False
    watched = _Watched(sparse.lib())
    with monkeypatch.context() as m:
        m.setattr(sparse, "lib", lambda: watched)
        got, got_len = sparse.build_sparse_list_decode(q, codes, norms, allowed, sink, window, M)
    base = got.shape[2] - M
    assert ("socket_finish_list" in watched.called) == (base > sparse._LONG_BASE)
    assert ("socket_select_list_allowed" in watched.called) == (base <= sparse._LONG_BASE)
    want, want_len = sparse._build_with_torch(q, codes, norms, allowed, sink, window, M)
    assert torch.equal(got, want) and torch.equal(got_len, want_len)
