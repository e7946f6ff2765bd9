"""A portion of more chunks than a grid's second dimension holds, in one call of the library."""
import pytest
import torch

from tests.test_hybrid_gpu import _recurrence

pytestmark = pytest.mark.gpu


def test_more_chunks_than_the_grids_y(dev, monkeypatch):
    """The whole portion in one scan gives the bits that scans of 2048 tokens give, whose chunks are the same."""
    from socket_amd import layer_ops
    from socket_amd.mixers import RecurrenceSpec as R, StepContext
    T = 65535 * 64 + 33                               # 65536 chunks, the last of 33 tokens
    br, cols, _ = _recurrence(dev, torch.bfloat16, R(1, 1, 16, 16, 8, False, decay="sigmoid_root", tau=8.0, gate="silu"), 1)
    proj = torch.randn(1, T, cols.total, generator=torch.Generator(dev).manual_seed(2), device=dev, dtype=torch.bfloat16)
    got = []
    for segment in (T, layer_ops.SCAN_SEGMENT):
        monkeypatch.setattr(layer_ops, "SCAN_SEGMENT", segment)
        br.alloc_state(1, T, torch.bfloat16, dev)
        out = br.heads(proj, StepContext(0, None, {}))
        got.append((out, br.state.s.clone()))
    assert torch.isfinite(got[0][0]).all()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
