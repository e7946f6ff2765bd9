"""The list builder and the attention over its list by the native step against the way through Python (which a function mode
takes): every type, odd sizes, windows and sinks at their ends, strided operands, several workgroups to a row, and what only
Python takes or refuses."""
import pytest
import torch

from socket_amd import _lib
from socket_amd.socket_kernels import sparse_attention_fwd
from socket_amd.sparse import build_sparse_list_decode

pytestmark = pytest.mark.gpu
DEV = "cuda"


class Watch(torch.overrides.TorchFunctionMode):
    """Sees torch's functions, so that nothing goes past it by address."""

    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def operands(B, H, Hkv, L, R, T, D, dtype, norm_dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    probs = torch.softmax(2 * torch.randn(B, H, L, R, generator=g, device=DEV), -1).to(dtype)
    codes = torch.randint(0, R, (B, H, L, T), generator=g, device=DEV).to(torch.int16)
    norms = (torch.rand(B, H, T, generator=g, device=DEV) + 0.5).to(norm_dtype)
    allowed = torch.rand(B, H, T, generator=g, device=DEV) < 0.9
    q = torch.randn(B, H, D, generator=g, device=DEV).to(dtype)
    k, v = (torch.randn(B, Hkv, T, D, generator=g, device=DEV).to(dtype) for _ in range(2))
    return (probs, codes, norms, allowed), (q, k, v)


def natively(ops, qkv, sink, window, M):
    """What the native step by itself makes of the operands: their list, its lengths and the attention, or None."""
    from socket_amd import sparse
    host, stream = _lib.host(), _lib.stream_ptr(qkv[0].device)
    lists = host.build_list(*ops, sink, window, M, sparse._LONG_BASE - 1, _lib.SOCKET_TOPK_MAX_M, sparse._select_workspace, stream)
    return lists and (*lists, host.sparse_attention(*qkv, *lists, stream))


def both(ops, qkv, sink, window, M, taken=True):
    direct = natively(ops, qkv, sink, window, M)
    lists = build_sparse_list_decode(*ops, sink, window, M)
    out = sparse_attention_fwd(*qkv, *lists)
    with Watch():
        want_lists = build_sparse_list_decode(*ops, sink, window, M)
        want = sparse_attention_fwd(*qkv, *want_lists)
    assert type(lists) is tuple and torch.equal(lists[0], want_lists[0]) and torch.equal(lists[1], want_lists[1])
    assert lists[0].dtype == lists[1].dtype == torch.int32 and out.dtype == qkv[0].dtype
    assert torch.equal(out, want)
    assert (direct is not None) == taken
    if taken:
        assert type(direct[2]) is torch.Tensor
        assert torch.equal(direct[0], want_lists[0]) and torch.equal(direct[1], want_lists[1]) and torch.equal(direct[2], want)


@pytest.mark.parametrize("dtype,norm_dtype", [(torch.bfloat16, torch.float16), (torch.float32, torch.float32), (torch.float16, torch.bfloat16)])
@pytest.mark.parametrize("B,H,Hkv,L,R,T,D,sink,window,M", [
    (1, 1, 1, 1, 4, 1, 16, 0, 0, 5), (2, 6, 2, 5, 32, 131, 64, 4, 16, 20), (1, 4, 4, 8, 256, 1000, 128, 1000, 7, 2000),
    (1, 2, 1, 3, 64, 70001, 32, 20, 0, 700), (3, 8, 4, 4, 128, 517, 128, 0, 600, 1),
    (1, 2, 2, 2, 16, 5000, 64, 96, 4000, 9), (1, 2, 2, 2, 16, 5000, 64, 96, 4001, 9),
    (1, 2, 2, 2, 16, 30000, 64, 96, 24479, 9), (1, 2, 2, 2, 16, 30000, 64, 96, 24480, 9)])      # (at and past the entries that it takes)
def test_same_as_through_python(dtype, norm_dtype, B, H, Hkv, L, R, T, D, sink, window, M):
    ops, qkv = operands(B, H, Hkv, L, R, T, D, dtype, norm_dtype, T)
    both(ops, qkv, sink, window, M, taken=sink + window < 24576)


def test_strided_rows_and_lists():
    ops, (q, k, v) = operands(2, 4, 2, 4, 64, 300, 64, torch.bfloat16, torch.float16, 1)
    wide = torch.randn(2, 300, 2, 128, device=DEV).bfloat16()
    qkv = (torch.randn(2, 8, 64, device=DEV).bfloat16()[:, ::2], wide[..., :64].transpose(1, 2), wide[..., 64:].transpose(1, 2))
    both(ops, qkv, 4, 8, 30)
    lists, lens = build_sparse_list_decode(*ops, 4, 8, 30)
    padded = torch.full((2, 4, 50), -1, dtype=torch.int32, device=DEV)
    padded[..., :42] = lists
    assert torch.equal(sparse_attention_fwd(q, k, v, padded[..., :42], lens), sparse_attention_fwd(q, k, v, lists, lens))


def test_what_goes_through_python():
    ops, (q, k, v) = operands(1, 4, 2, 4, 64, 200, 64, torch.bfloat16, torch.float16, 2)
    want = build_sparse_list_decode(*ops, 2, 4, 16)
    probs, codes, norms, allowed = ops
    host = _lib.host()

    def native(*o, sink=2, window=4, M=16):
        return host.build_list(*o, sink, window, M, 24576, 4096, lambda *_: None, _lib.stream_ptr(q.device))

    spread = torch.stack([norms, norms], -1)[..., 0]
    for o in ((probs, codes.int(), norms, allowed), (probs, codes, spread, allowed), (torch.nn.Parameter(probs), codes, norms, allowed)):
        got = build_sparse_list_decode(*o, 2, 4, 16)
        assert torch.equal(got[0], want[0])
    assert native(probs, codes.int(), norms, allowed) is None and native(probs, codes, spread, allowed) is None
    assert native(*ops, window=True) is None and native(*ops, M=0) is None and native(*ops, M=1 << 70) is None
    assert native(probs, codes[:, :2], norms, allowed) is None and native(probs.cpu(), codes, norms, allowed) is None
    got = build_sparse_list_decode(*ops, 2, 4, 0)
    assert got[0].shape[-1] == 6
    with pytest.raises(AssertionError):
        build_sparse_list_decode(probs, codes, norms, allowed.int(), 2, 4, 16)
    with pytest.raises(AssertionError):
        sparse_attention_fwd(q, k.float(), v, *want)
    with pytest.raises(AssertionError):
        sparse_attention_fwd(q.cpu(), k, v, *want)
    assert sparse_attention_fwd(q, k, v, want[0][..., :0], want[1]).isnan().all()
    assert torch.equal(sparse_attention_fwd(q, k, v, want[0].long(), want[1].long()), sparse_attention_fwd(q, k, v, *want))
    with pytest.raises(RuntimeError):      # (the library wants rows on 16-byte boundaries)
        sparse_attention_fwd(torch.randn(1, 4 * 64 + 1, device=DEV).bfloat16()[:, 1:].view(1, 4, 64), k, v, *want)
    assert not sparse_attention_fwd(q.requires_grad_(), k, v, *want).requires_grad


@pytest.mark.parametrize("T", [3000, 70001])      # (one workgroup to a row, and several, which need the workspace)
def test_on_a_side_stream_and_captured(T):
    ops, qkv = operands(1, 2, 1, 3, 64, T, 64, torch.bfloat16, torch.float16, 7)
    want = natively(ops, qkv, 4, 64, 300)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = build_sparse_list_decode(*ops, 4, 64, 300)
        got = (*got, sparse_attention_fwd(*qkv, *got))
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    q = qkv[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        lists = build_sparse_list_decode(*ops, 4, 64, 300)
        out = sparse_attention_fwd(q, *qkv[1:], *lists)
    for turn in range(4):
        ops[0].copy_(torch.roll(ops[0], 1, -1))
        q.copy_(torch.roll(q, 1, -1))
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        want = natively(ops, (q, *qkv[1:]), 4, 64, 300)
        assert torch.equal(lists[0], want[0]) and torch.equal(lists[1], want[1]) and torch.equal(out, want[2])
