"""Rows that start on any element: the reference's operand layout at contexts that are a multiple of nothing."""
import pytest
import torch

from socket_amd import sparse
from socket_amd._lib import check, dtype_enum, lib, ptr, stream_ptr

pytestmark = pytest.mark.gpu


def _collide(q, codes, allowed, v, out):
    B, H, L, R = q.shape
    check("socket_soft_hash_collision", lib().socket_soft_hash_collision_typed(
        ptr(q), dtype_enum(q.dtype), ptr(codes), ptr(allowed), ptr(v), dtype_enum(v.dtype), ptr(out), B, H, L, R, codes.shape[3],
        stream_ptr(q.device)))


@pytest.mark.parametrize("B,H,L,R,T,qt,vt,shift", [
    (1, 2, 5, 64, 1, torch.float32, torch.float16, 0),           # fewer tokens than a thread's eight
    (1, 3, 5, 64, 7, torch.bfloat16, torch.float32, 0),
    (2, 3, 7, 256, 8, torch.float16, torch.float16, 0),          # exactly eight, odd bases
    (1, 3, 7, 256, 9, torch.float32, torch.bfloat16, 1),         # the second thread owns one
    (2, 5, 60, 1024, 2051, torch.float32, torch.float16, 3),     # two table slices: sums wait in the output between them
    (1, 32, 60, 1024, 8195, torch.float32, torch.float32, 0),    # several tiles to a workgroup
    (2, 28, 48, 1024, 20881, torch.bfloat16, torch.float16, 5),  # codes loaded past the caches
    (1, 32, 60, 1024, 16383, torch.bfloat16, torch.float16, 1),  # two tokens to a lane, one short of every lane's two
    (1, 32, 7, 1024, 16385, torch.float32, torch.bfloat16, 0),   # ... one more: four to a lane
    (1, 32, 60, 1024, 24577, torch.float32, torch.float16, 1),   # ... and one past the last of those
    (3, 7, 3, 16, 131, torch.bfloat16, torch.bfloat16, 0),       # a tile and three tokens
    (1, 2, 3, 65536, 4101, torch.float32, torch.float16, 0),     # a table that exceeds LDS
])
def test_collision_scores_of_odd_rows(B, H, L, R, T, qt, vt, shift):
    """Bit for bit the sequential fp32 sum, masked, for rows and bases on no boundary; codes outside [0, R) add nothing;
    nothing is written outside the scores."""
    dev = "cuda"
    g = torch.Generator(device=dev).manual_seed(T)
    q = torch.rand(B, H, L, R, generator=g, device=dev).to(qt)
    n = B * H * T

    def at(flat, shape):      # (the values `shift` elements into an allocation)
        whole = torch.empty(flat.numel() + shift, dtype=flat.dtype, device=dev)
        whole[shift:] = flat
        return whole[shift:].view(shape)

    codes = at(torch.randint(-2, min(R + 2, 32767), (n * L,), generator=g, device=dev).to(torch.int16), (B, H, L, T))
    allowed = at(torch.rand(n, generator=g, device=dev) < 0.8, (B, H, T))
    v = at((torch.rand(n, generator=g, device=dev) * 4).to(vt), (B, H, T))
    buf = torch.full((n + shift + 16,), 7.0, device=dev)
    out = buf[shift:shift + n].view(B, H, T)
    _collide(q, codes, allowed, v, out)
    want = torch.zeros(B, H, T, device=dev)
    for l in range(L):
        c = codes[:, :, l].long()
        want += torch.gather(q[:, :, l].float(), 2, c.clamp(0, R - 1)).masked_fill((c < 0) | (c >= R), 0.0)
    want = (want * v.float()).masked_fill(~allowed, float("-inf"))
    assert torch.equal(out, want)
    assert (buf[:shift] == 7.0).all() and (buf[shift + n:] == 7.0).all()


@pytest.mark.parametrize("T,M,shift", [(5, 3, 1), (4135, 129, 0), (8193, 300, 3), (20881, 652, 0), (49157, 1024, 2), (131075, 2048, 1)])
def test_selection_from_odd_rows(T, M, shift):
    """The list of a stable descending sort, from rows of odd pitch that start on any float, some scores minus infinity."""
    dev, H = "cuda", 5
    g = torch.Generator(device=dev).manual_seed(T)
    whole = torch.randn(H * T + shift, generator=g, device=dev).exp_()
    scores = whole[shift:].view(1, H, T)
    scores[:, 1:3].masked_fill_(torch.rand(1, 2, T, generator=g, device=dev) < 0.5, float("-inf"))
    scores[:, 3, :] = scores[:, 3, :].round()      # (many equal ones)
    lists, lens = sparse.select_list(scores, 0, 0, M, write_base=False)
    assert (lens == M).all()
    assert torch.equal(lists.long(), torch.sort(scores, dim=-1, descending=True, stable=True).indices[..., :M])


@pytest.mark.parametrize("B,H,T,M,sink,window,kept", [
    (1, 4, 5, 5, 2, 2, 0.5),                # more asked for than are allowed
    (2, 7, 4135, 129, 20, 20, 0.5),
    (1, 8, 8192, 700, 0, 0, 0.05),          # fewer allowed than are asked for: masked ones, mostly of one run, fill the list
    (1, 8, 8193, 300, 4, 64, 0.9),          # threshold from a sample
    (2, 5, 20881, 652, 4, 64, 0.02),        # ... of which little is allowed
    (1, 6, 49157, 1024, 4, 64, 0.6),        # a row shared between workgroups
    (1, 3, 9000, 128, 3, 9000, 0.7),        # a window that is the whole row
])
def test_masked_lists(B, H, T, M, sink, window, kept):
    """The list builder's masked selection against the unmasked one with torch's masking around it; the second row of every
    sequence has nothing allowed, the third everything."""
    dev, L, R = "cuda", 4, 64
    g = torch.Generator(device=dev).manual_seed(T + M)
    q = torch.rand(B, H, L, R, generator=g, device=dev)
    codes = torch.randint(0, R, (B, H, L, T), generator=g, device=dev).to(torch.int16)
    norms = (torch.rand(B, H, T, generator=g, device=dev) + 0.1).half()
    allowed = torch.rand(B, H, T, generator=g, device=dev) < kept
    allowed[:, 0, T // 2:] = False
    allowed[:, 1], allowed[:, 2] = False, True
    got, got_len = sparse.build_sparse_list_decode(q, codes, norms, allowed, sink, window, M)
    want, want_len = sparse._build_with_torch(q, codes, norms, allowed, sink, window, min(M, T))
    assert torch.equal(got, want) and torch.equal(got_len, want_len)
