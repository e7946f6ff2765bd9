"""The scorer on the reference's own operands: codes inside and outside the table, and tiles that its launches deal out evenly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scores(probs, codes, allowed, norms):
    """The definition, summed over the tables in order in float32."""
    B, H, L, T = codes.shape
    R = probs.shape[-1]
    s = torch.zeros(B, H, T, device=codes.device)
    for l in range(L):
        c = codes[:, :, l].long()
        inside = (c >= 0) & (c < R)
        e = probs[:, :, l].float().gather(-1, c.clamp(0, R - 1))
        s += torch.where(inside, e, torch.zeros_like(e))
    return torch.where(allowed, s * norms.float(), torch.full_like(s, float("-inf")))


def _run(probs, codes, allowed, norms):
    from socket_amd._lib import check, dtype_enum, lib, ptr, stream_ptr
    B, H, L, T = codes.shape
    out = torch.full((B, H, T), float("nan"), device=codes.device)
    check("scores", lib().socket_soft_hash_collision_typed(
        ptr(probs), dtype_enum(probs.dtype), ptr(codes), ptr(allowed), ptr(norms), dtype_enum(norms.dtype), ptr(out), B, H, L,
        probs.shape[-1], T, stream_ptr(codes.device)))
    return out


def _operands(B, H, L, T, R, dtype, seed):
    dev, g = "cuda", torch.Generator(device="cuda").manual_seed(seed)
    probs = torch.rand(B, H, L, R, generator=g, device=dev).to(dtype)
    codes = torch.randint(0, min(R, 32768), (B, H, L, T), generator=g, device=dev).to(torch.int16)
    allowed = torch.rand(B, H, T, generator=g, device=dev) < 0.9
    return probs, codes, allowed, torch.rand(B, H, T, generator=g, device=dev).half()


# (R at and past the largest code; T: two, four and eight tokens a lane; "strays": lanes, whole waves, every code)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("R", [1, 3, 256, 1024, 32767, 32768, 40000])
@pytest.mark.parametrize("T", [8, 999, 5001, 33001])
def test_codes_outside_the_table_add_nothing(dtype, R, T):
    B, H, L = 1, (3 if T < 9000 else 16), 7
    probs, codes, allowed, norms = _operands(B, H, L, T, R, dtype, R + T)
    assert torch.equal(_run(probs, codes, allowed, norms), _scores(probs, codes, allowed, norms))
    strays = torch.tensor([-1, -32768, 32767, min(R, 32767), min(R + 1, 32767)], dtype=torch.int16, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(T)
    for share in (0.001, 0.3, 1.0):
        pick = torch.rand(codes.shape, generator=g, device="cuda") < share
        c = torch.where(pick, strays[torch.randint(0, 5, codes.shape, generator=g, device="cuda")], codes)
        c[:, :, :, T // 2:T // 2 + 600] = codes[:, :, :, T // 2:T // 2 + 600]      # (waves without any beside those with some)
        assert torch.equal(_run(probs, c, allowed, norms), _scores(probs, c, allowed, norms))


# tiles of whole waves over the CUs of a row: the last one short, one wave long, or missing; two slices of tables; rows that
# two workgroups each take; more tokens than one round holds
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,H,L,T,R", [(1, 28, 48, 33000, 1024), (1, 16, 60, 60001, 1024), (2, 28, 12, 20001, 1024), (1, 5, 60, 262145, 256),
                                       (1, 128, 4, 16385, 1024), (1, 200, 3, 4609, 1024), (3, 100, 3, 9001, 512), (1, 1, 2, 2049, 1024),
                                       (1, 32, 60, 4097, 1024)])
def test_tiles(dtype, B, H, L, T, R):
    probs, codes, allowed, norms = _operands(B, H, L, T, R, dtype, T)
    assert torch.equal(_run(probs, codes, allowed, norms), _scores(probs, codes, allowed, norms))


# codes past what a cache keeps from call to call, four and eight tokens a lane, also with some outside the table
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,L,T,R", [(32, 130, 24575, 64), (56, 48, 40003, 256)])
def test_streamed_codes(dtype, H, L, T, R):
    probs, codes, allowed, norms = _operands(1, H, L, T, R, dtype, T)
    assert codes.numel() * 2 > 192 << 20
    assert torch.equal(_run(probs, codes, allowed, norms), _scores(probs, codes, allowed, norms))
    codes[:, :, ::7, ::1013] = -1
    assert torch.equal(_run(probs, codes, allowed, norms), _scores(probs, codes, allowed, norms))
