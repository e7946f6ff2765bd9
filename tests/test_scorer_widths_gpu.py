"""The operator scorer at every width of its workgroups: tables that fill a CU's LDS and tables that share it, one slice and
several, 16-byte and 2-byte code loads, on both sides of each line.  Sums run over the tables in order in 32 bits, so the
scores are equal bit by bit to the same sums by torch."""
import pytest
import torch

from socket_amd._lib import check, dtype_enum, lib, ptr, stream_ptr

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,L,R,T", [(2, 16, 5000, 2048), (2, 16, 5000, 2049), (2, 16, 5000, 2056), (2, 16, 5000, 2816), (2, 16, 5000, 2817),
                                     (2, 60, 1024, 4096), (2, 60, 1024, 4104), (2, 60, 1024, 4608), (2, 60, 1024, 4616), (1, 60, 1024, 6145),
                                     (30, 60, 1024, 9000),
                                     (33, 16, 5000, 16391), (33, 16, 5000, 32770), (65, 8, 5000, 32768), (3, 7, 200, 2050), (3, 7, 200, 9000),
                                     (90, 4, 300, 6200)])
def test_scores_bit_by_bit(H, L, R, T, dt):
    g = torch.Generator(device=DEV).manual_seed(T)
    q = torch.rand(1, H, L, R, generator=g, device=DEV).to(dt)
    codes = torch.randint(0, R, (1, H, L, T), generator=g, device=DEV, dtype=torch.int16)
    norms = torch.rand(1, H, T, generator=g, device=DEV).half()
    allowed = torch.rand(1, H, T, generator=g, device=DEV) < 0.9
    got = torch.empty(1, H, T, device=DEV)
    check("socket_soft_hash_collision_typed", lib().socket_soft_hash_collision_typed(
        ptr(q), dtype_enum(dt), ptr(codes), ptr(allowed), ptr(norms), dtype_enum(norms.dtype), ptr(got), 1, H, L, R, T, stream_ptr()))
    want = torch.zeros(1, H, T, device=DEV)
    for l in range(L):
        want += torch.gather(q[:, :, l].float(), 2, codes[:, :, l].long())
    want = (want * norms.float()).masked_fill(~allowed, -torch.inf)
    assert torch.equal(got, want)
