"""Modules of the decoder under torch's tracers: what a tracer records is torch operations, never an output that a
kernel launch it cannot see would have filled."""

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

from socket_amd import _lib, decode_ops, layer_ops
from socket_amd.model import FeedForward, ModelArgs, RMSNorm, Transformer


class Passing(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class Seeing(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def in_mode(mode):
    def trace(f, x):
        with mode():
            f(x)
    return trace


TRACERS = {
    "jit": lambda f, x: torch.jit.trace(f, (x,), check_trace=False),
    "make_fx": lambda f, x: make_fx(f)(x),
    "make_fx_fake": lambda f, x: make_fx(f, tracing_mode="fake")(x),
    "make_fx_symbolic": lambda f, x: make_fx(f, tracing_mode="symbolic")(x),
    "make_fx_pre_dispatch": lambda f, x: make_fx(f, pre_dispatch=True)(x),
    "compile": lambda f, x: torch.compile(f, backend="eager", fullgraph=True),
}
MODES = {
    "vmap": lambda f, x: torch.vmap(f)(x[None]),
    "jvp": lambda f, x: torch.func.jvp(f, (x,), (x,)),
    "dispatch": in_mode(Passing),
    "function": in_mode(Seeing),
}


def norm(device, dtype):
    m = RMSNorm(64).to(device, dtype)
    m.weight.data.uniform_(0.5, 1.5)
    return m


def feed_forward(device, dtype):
    torch.manual_seed(0)
    return FeedForward(ModelArgs(dim=64, n_head=2, intermediate_size=128)).to(device, dtype)


@pytest.mark.parametrize("make", [norm, feed_forward])
def test_symbolic_trace_and_script_on_the_host(make):
    m, x = make("cpu", torch.float32), torch.randn(3, 5, 64)
    for traced in (torch.fx.symbolic_trace(m), torch.jit.script(m)):
        assert torch.equal(traced(x), m(x))


@pytest.mark.parametrize("name", [n for n in TRACERS if n != "compile"] + list(MODES))
def test_every_tracer_is_seen(name):
    seen = []

    def f(x):
        seen.append(_lib.observed())
        return x * 2

    assert not _lib.observed()
    with torch.no_grad():
        ({**TRACERS, **MODES}[name])(f, torch.ones(4))
    assert seen and all(seen)
    with torch.device("cpu"):
        assert not _lib.observed()


def test_tensors_of_two_devices_are_told_apart():
    a, b = torch.ones(2), torch.ones(2, device="meta")
    assert _lib.one_device((a, a)) and _lib.one_device((b,)) and not _lib.one_device((a, b))


@pytest.mark.gpu
def test_a_kernel_takes_no_operand_of_another_device():
    x = torch.ones(4, 64, device="cuda")
    assert decode_ops.pointwise_fits(x, x) and not decode_ops.pointwise_fits(x, x.cpu())


@pytest.mark.gpu
@pytest.mark.parametrize("make", [norm, feed_forward])
@pytest.mark.parametrize("name", ["jit", "make_fx", "make_fx_pre_dispatch", "compile", "fx", "script"])
def test_traced_modules_compute_on_the_device(name, make):
    m = make("cuda", torch.bfloat16)
    x, y = (torch.randn(2, 9, 64, device="cuda").bfloat16() for _ in range(2))
    with torch.no_grad():
        if name == "fx":
            traced = torch.fx.symbolic_trace(m)
        elif name == "script":
            traced = torch.jit.script(m)
        else:
            traced = TRACERS[name](m, x)
        want = m(y)
        torch.empty_like(want).fill_(float("nan"))      # (memory that an output nothing fills would take)
        assert torch.equal(traced(y), want)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["jit", "make_fx"])
def test_a_traced_prompt_is_the_prompt(name):
    torch.manual_seed(1)
    model = Transformer(ModelArgs(block_size=64, vocab_size=96, n_layer=2, n_head=2, dim=128, intermediate_size=128,
                                  L=4, K=4, R=16)).to("cuda", torch.bfloat16).eval().requires_grad_(False)
    with torch.device("cuda"):
        model.setup_caches(1, 64)
    ids, more = (torch.randint(0, 96, (1, 24), device="cuda") for _ in range(2))
    pos = torch.arange(24, device="cuda")
    with torch.no_grad():
        def f(t):
            return model(t, pos, pos0=0)

        traced = TRACERS[name](f, ids)
        want = model(more, pos, pos0=0)
        got = traced(more)
        # (torch's attention in the traced form: weights and result rounded elsewhere)
        assert (got.float() - want.float()).norm() < 0.02 * want.float().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(TRACERS) + list(MODES))
def test_no_kernel_stands_for_torch_operations_there(name):
    q = torch.randn(1, 8, 4, 64, device="cuda").bfloat16()
    cache = torch.zeros(1, 4, 16, 64, device="cuda").bfloat16()
    freqs = torch.zeros(8, 32, 2, device="cuda").bfloat16()
    qkv = torch.zeros(1, 8, 12 * 64, device="cuda").bfloat16()
    seen = []

    def f(x):
        seen.append(decode_ops.pointwise_fits(x, x) or layer_ops.prompt_attend_fits(q, q, q)
                    or decode_ops.rope_rows_fits(qkv, freqs, cache, cache))
        return x * 2

    with torch.no_grad():
        assert decode_ops.pointwise_fits(q, q) and layer_ops.prompt_attend_fits(q, q, q)
        assert decode_ops.rope_rows_fits(qkv, freqs, cache, cache)
        out = ({**TRACERS, **MODES}[name])(f, torch.ones(4, device="cuda"))
        if name == "compile":
            out(torch.ones(4, device="cuda"))
    assert seen and not any(seen)
