"""How far the chunked recurrences are from float64: the running sums of the log decays, which every exponent of a chunk is
a difference of, are what their 32-bit precision rests on."""
import pytest
import torch

from tests.test_hybrid_gpu import _rand, _recurrence, _recurrence_oracle

pytestmark = pytest.mark.gpu


def _off(got, want):
    return float((got.cpu().double() - want).norm() / want.norm())


@pytest.mark.parametrize("name,shift,what,bound", [
    # An entry of a block's running sums is rounded at the sum's magnitude, 2^-24 x 60 at most.  Summed row after row, two
    # neighbours differ by one such rounding; halves summed apart and put together afterwards, by two.  Means over the three
    # seeds 2.4e-7, 2.1e-7 and 2.5e-7 in order, 4.9e-7, 3.0e-7 and 3.4e-7 in halves; the bounds lie between.
    ("delta", 2.0, "state", 3.2e-7),
    ("delta", 0.0, "state", 2.5e-7),
    ("gla", -2.0, "out", 2.9e-7),
])
def test_decays_are_summed_in_order(dev, name, shift, what, bound):
    from socket_amd.mixers import RecurrenceSpec as R, StepContext
    spec = (R(2, 1, 128, 128, 16, True, 4, True, gate_rank=16) if name == "delta"
            else R(2, 2, 64, 128, 12, False, decay="sigmoid_root", tau=2.0, gate="silu"))
    T, errors = 400, []
    for seed in range(3):
        br, cols, vals = _recurrence(dev, torch.float32, spec, seed, shift)
        proj = _rand(torch.Generator().manual_seed(seed + 50), 1, T, cols.total)
        out, state = _recurrence_oracle(spec, cols, vals, proj[0])
        br.alloc_state(1, T, torch.float32, dev)
        got = br.heads(proj.to(dev, torch.float32), StepContext(0, None, {}))
        errors.append(_off(br.state.s[0], state) if what == "state" else _off(got[0], out))
    assert sum(errors) / len(errors) < bound, errors
