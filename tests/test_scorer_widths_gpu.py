"""The operator scorer in each of its forms: two and four tokens to a lane where rows are short for their number of CUs,
eight with workgroups of 256, 512 and 1024 lanes, tables in LDS in one slice and several or past it, on both sides of each
line.  Sums run over the tables in order in 32 bits, so the scores are equal bit by bit to the same sums by torch."""
import pytest
import torch

from socket_amd._lib import check, dtype_enum, lib, ptr, stream_ptr

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (lines for 256 CUs)
_TWO = [(2, 16, 5000, 2048), (2, 16, 5000, 2049), (2, 16, 5000, 2056), (2, 16, 5000, 2816), (2, 16, 5000, 2817), (2, 60, 1024, 4096),
        (2, 60, 1024, 4104), (2, 60, 1024, 4608), (2, 60, 1024, 4616), (1, 60, 1024, 6145), (30, 60, 1024, 9000), (3, 7, 200, 2050),
        (3, 7, 200, 9000), (32, 8, 1024, 16384), (256, 3, 300, 2048)]
_FOUR = [(32, 8, 1024, 16385), (33, 16, 5000, 16391), (32, 60, 1024, 24576), (90, 4, 300, 6144), (256, 3, 300, 3072)]
_256 = [(257, 6, 200, 8), (257, 6, 200, 2041), (300, 60, 1024, 2048)]
_512 = [(32, 60, 1024, 24577), (32, 8, 5000, 32768), (65, 8, 5000, 9217), (64, 8, 1024, 16383), (128, 4, 300, 6145), (128, 4, 300, 8192),
        (90, 4, 300, 6200)]
_1024 = [(32, 8, 1024, 32769), (33, 16, 5000, 32770), (65, 8, 5000, 32768), (257, 6, 200, 2049), (256, 4, 300, 4099), (128, 4, 300, 8193)]
_PAST_LDS = [(2, 3, 65000, 2047), (2, 3, 65000, 4608), (2, 3, 65000, 9001)]      # (in float32; bfloat16 tables of that size fit)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,L,R,T", _TWO + _FOUR + _256 + _512 + _1024 + _PAST_LDS)
def test_scores_bit_by_bit(H, L, R, T, dt):
    g = torch.Generator(device=DEV).manual_seed(T)
    q = torch.rand(1, H, L, R, generator=g, device=DEV).to(dt)
    codes = torch.randint(0, min(R, 32768), (1, H, L, T), generator=g, device=DEV, dtype=torch.int16)
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
