"""Which rows the native append takes, form by form, against the same conditions written out in Python, and what it then
writes against torch's copies and the separate hash, bit for bit."""
import pytest
import torch
from torch.overrides import TorchFunctionMode

from socket_amd import _lib, hash_cache

DEV = "cuda"


class Mode(TorchFunctionMode):
    def __torch_function__(self, fn, types, args=(), kwargs=None):
        return fn(*args, **(kwargs or {}))


class Other(torch.Tensor):
    pass


def takes(c, k, v):
    kc, vc = c.k_cache, c.v_cache
    if any(type(t) not in (torch.Tensor, torch.nn.Parameter) or not t.is_cuda for t in (k, v)):
        return False
    step = 16 // kc.element_size()
    return (k.dtype == v.dtype == kc.dtype and k.shape == v.shape and k.shape[2:] == (kc.shape[1], kc.shape[3]) and k.shape[1] > 0
            and k.shape[3] % 8 == 0 and k.shape[3] <= 128 and kc.is_contiguous() and vc.is_contiguous()
            and all(t.stride(3) == 1 and all(s % step == 0 for s in t.stride()[:3]) and t.data_ptr() % 16 == 0 for t in (k, v)))


def forms(c, dt, S=5):
    """Pairs of rows (k, v) in every form an append may be given."""
    B, H, _, D = c.k_cache.shape
    new = lambda *shape, dtype=dt: torch.randn(*shape, device=DEV).to(dtype)
    yield "plain", new(B, S, H, D), new(B, S, H, D)
    yield "no rows", new(B, 0, H, D), new(B, 0, H, D)
    yield "heads first", new(B, H, S, D).transpose(1, 2), new(B, S, H, D)
    yield "views of one projection", *new(B, S, 2 * H, D).split(H, 2)
    yield "expanded over heads", new(B, S, 1, D).expand(B, S, H, D), new(B, S, H, D)
    yield "every second dimension", new(B, S, H, 2 * D)[..., ::2], new(B, S, H, D)
    yield "odd row stride", new(B, S, H, D + 1)[..., :D], new(B, S, H, D)
    yield "odd value stride", new(B, S, H, D), new(B, S, H, D + 1)[..., :D]
    yield "off by one element", new(B * S * H * D + 1)[1:].view(B, S, H, D), new(B, S, H, D)
    yield "off by 16 bytes", new(B * S * H * D + 8)[16 // c.k_cache.element_size():][:B * S * H * D].view(B, S, H, D), new(B, S, H, D)
    yield "another type", new(B, S, H, D, dtype=torch.float64), new(B, S, H, D)
    yield "values of another type", new(B, S, H, D), new(B, S, H, D, dtype=torch.float64)
    yield "one parameter", torch.nn.Parameter(new(B, S, H, D)), new(B, S, H, D)
    yield "a subclass", new(B, S, H, D).as_subclass(Other), new(B, S, H, D)
    yield "host memory", new(B, S, H, D).cpu(), new(B, S, H, D)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [8, 20, 64, 128])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_native_append_takes_and_writes_what_it_should(dt, D):
    B, H, pos0 = 2, 3, 6
    torch.manual_seed(D)
    planes = torch.randn(60, 10, D, device=DEV)
    taken = 0
    for name, k, v in forms(hash_cache.SocketHashCache(B, 24, H, D, 60, 10, dtype=dt, device=DEV), dt):
        one, two = (hash_cache.SocketHashCache(B, 24, H, D, 60, 10, dtype=dt, device=DEV) for _ in range(2))
        two._native_append = lambda *a: -1      # torch's copies, then the hash
        for c in (one, two):
            c.set_planes(planes)
        fits = one._append_fits(k, v)
        assert fits == takes(one, k, v), name
        with Mode():
            assert not one._append_fits(k, v), name
        if not fits:
            continue
        taken += 1
        for c in (one, two):
            c.append(pos0, k, v)
        for a, b in zip((one.k_cache, one.v_cache, one.codes, one.v_norm, one.lens), (two.k_cache, two.v_cache, two.codes, two.v_norm, two.lens)):
            assert torch.equal(a, b), name
    assert taken == (0 if D % 8 else 6)


@pytest.mark.gpu
def test_native_append_asks_the_cache_too():
    make = lambda: hash_cache.SocketHashCache(2, 24, 3, 64, 60, 10, device=DEV)
    rows = torch.randn(2, 5, 3, 64, device=DEV).bfloat16()
    planes = torch.randn(60, 10, 64, device=DEV)
    for name in ("k_cache", "v_cache", "codes", "v_norm", "lens"):
        c = make()
        c.set_planes(planes)
        assert c._append_fits(rows, rows)
        whole = getattr(c, name)
        setattr(c, name, torch.zeros(*whole.shape, 2, dtype=whole.dtype, device=DEV)[..., 0])
        assert not c._append_fits(rows, rows), name
    c = make()
    c.set_planes(planes)
    c.v_cache = c.v_cache.half()
    assert not c._append_fits(rows, rows)
    with pytest.raises(RuntimeError):      # a sparse tensor has no strides
        make_sparse = make()
        make_sparse.set_planes(planes)
        make_sparse.append(0, rows.to_sparse(), rows)


def test_native_call_refuses_without_a_device():
    z = torch.zeros(2, 3, 4, 8)
    call = _lib.host().cache_append
    assert call(*[z] * 8, 0, 1, 1, 8, 0, False) == -1
    assert call(None, *[z] * 7, 0, 1, 1, 8, 0, True) == -1
    with pytest.raises(TypeError):
        call(z)
    with pytest.raises(TypeError):
        call(*[z] * 8, "0", 1, 1, 8, 0, False)
