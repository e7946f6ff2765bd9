"""Read-outs of the chunked recurrences, which the scan takes a barrier behind the state: one, two, three and four chunks, a last
one of a single token, more row blocks than waves have, and read-outs with and without a state before them."""
import pytest
import torch

from tests import hybrid_models as hm
from tests.test_hybrid_gpu import _rand, _recurrence, _recurrence_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dk,delta", [(16, True), (64, True), (128, True), (144, True), (256, True), (16, False), (64, False), (128, False), (144, False)])
@pytest.mark.parametrize("chunks", [1, 2, 3, 4])
def test_read_outs_of_few_chunks(dev, dk, delta, chunks):
    from socket_amd.mixers import RecurrenceSpec as R, StepContext
    spec = (R(2, 1, dk, 48, 16, True, 4, True, gate_rank=16) if delta else
            R(2, 2, dk, 48, 12, False, decay="sigmoid_root", tau=8.0, gate="silu"))
    C = 64 if dk <= 128 else 32
    T = (chunks - 1) * C + (1 if chunks % 2 == 0 else C)
    br, cols, vals = _recurrence(dev, torch.float32, spec, dk + chunks, 0.0)
    proj = _rand(torch.Generator().manual_seed(T), 1, T + 5, cols.total)
    want, state = _recurrence_oracle(spec, cols, vals, proj[0])
    br.alloc_state(1, T + 5, torch.float32, dev)
    p = proj.to(dev, torch.float32)
    got = torch.cat([br.heads(p[:, :5], StepContext(0, None, {})), br.heads(p[:, 5:], StepContext(5, None, {}))], 1).cpu()
    # (as in test_recurrence_tiles_gpu.py: a few units of 2^-24 times the root of at most 256 products, and the norm's division)
    assert hm.rms_error(got[0], want) < 5e-5
    assert hm.rms_error(br.state.s[0].cpu().flatten(1), state.flatten(1)) < 2e-5
