"""Chunked recurrences where the preparation and the scan take another branch: odd and even numbers of chunks and a rest
beside full ones, V in LDS by itself or over what has been used, decays so strong that a diagonal tile takes its
exponents pair by pair, an odd number of state tiles."""
import pytest
import torch

from tests import hybrid_models as hm
from tests.test_hybrid_gpu import _rand, _recurrence, _recurrence_oracle

pytestmark = pytest.mark.gpu


def _specs():
    from socket_amd.mixers import RecurrenceSpec as R
    return {
        "delta_split_tiles": (R(2, 1, 128, 128, 16, True, 4, True, gate_rank=16), 8.0),
        "delta_some_split": (R(2, 2, 128, 64, 16, True, 2, True, gate_rank=16), 3.0),
        "delta_wide_values": (R(1, 1, 128, 256, 16, True, 4, True, gate_rank=16), 0.0),      # V over q
        "delta_seven_tiles": (R(1, 1, 112, 40, 16, True, 4, True, gate_rank=16), 1.0),
        "gla_split_tiles": (R(2, 2, 64, 128, 12, False, decay="sigmoid_root", tau=0.25, gate="silu"), -8.0),
        "gla_wide_values": (R(1, 1, 80, 256, 12, False, decay="sigmoid_root", tau=8.0, gate="silu"), 0.0),
        "gla_conv": (R(2, 1, 32, 32, 12, False, 6, True, decay="sigmoid_root", tau=8.0, gate="silu"), 0.0),   # more taps than are read at once
    }


@pytest.mark.parametrize("T", [64, 65, 128, 193, 320])
@pytest.mark.parametrize("name", ["delta_split_tiles", "delta_some_split", "delta_wide_values", "delta_seven_tiles",
                                  "gla_split_tiles", "gla_wide_values", "gla_conv"])
def test_chunks_against_one_token_at_a_time(dev, name, T):
    from socket_amd.mixers import StepContext
    spec, shift = _specs()[name]
    br, cols, vals = _recurrence(dev, torch.float32, spec, len(name) + T, shift)
    proj = _rand(torch.Generator().manual_seed(T), 2, T, cols.total)
    want = [_recurrence_oracle(spec, cols, vals, proj[b]) for b in range(2)]
    br.alloc_state(2, T, torch.float32, dev)
    first = 3 if T % 2 else 0                       # (a state and conv rows that the chunks start from)
    p = proj.to(dev, torch.float32)
    out = [br.heads(p[:, :first], StepContext(0, None, {}))] if first else []
    out.append(br.heads(p[:, first:], StepContext(first, None, {})))
    got = torch.cat(out, 1).cpu()
    assert torch.isfinite(got).all()
    # 32-bit products and sums over at most 256 channels and 64 tokens of a chunk: a few units of 2^-24 times the root of
    # their number, 1e-6, with a margin for the norm's division
    for b in range(2):
        assert hm.rms_error(br.state.s[b].cpu().flatten(1), want[b][1].flatten(1)) < 2e-5, b
    assert hm.rms_error(got, torch.stack([x[0] for x in want])) < 5e-5
