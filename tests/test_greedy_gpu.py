"""The end of a greedy decode step in one launch: the first of the greatest logits, and the position after it."""
import pytest
import torch

from socket_amd import decode_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [1, 15, 16, 19, 4095, 8200, 32000, 65537])
@pytest.mark.parametrize("pad", [0, 3, 8])              # (row strides with and without whole 16-byte pieces)
def test_against_argmax(dtype, V, pad):
    g = torch.Generator().manual_seed(V + pad)
    wide = torch.randn(6, V + pad, generator=g).to(dtype)
    wide[1, :V] = wide[1, :V].round()                     # many equal greatest values: the first of them
    wide[2, :V] = float("-inf")
    wide[3, V // 2] = float("nan")
    wide[3, V - 1] = float("nan")
    wide[4, :V] = -0.0
    wide[4, V // 3:V] = 0.0                               # (equal to -0)
    wide[5, V - 1] = float("inf")
    logits = wide.cuda()[:, :V]
    tok = torch.full((6, 1), -7, dtype=torch.int32, device="cuda")
    pos = torch.tensor([41], device="cuda")
    want = wide[:, :V].float().argmax(-1, keepdim=True).int()
    assert torch.equal(decode_ops.greedy_tokens(logits).cpu(), want)
    assert decode_ops.greedy_tokens(logits, out=tok, pos=pos) is tok
    assert torch.equal(tok.cpu(), want) and int(pos) == 42


def test_columns_and_other_types_take_the_general_way():
    x = torch.randn(50, 4, device="cuda")
    assert torch.equal(decode_ops.greedy_tokens(x.t()), x.argmax(0, keepdim=True).t().int())
    y = torch.randn(3, 50, device="cuda", dtype=torch.float64)
    assert torch.equal(decode_ops.greedy_tokens(y), y.argmax(-1, keepdim=True).int())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [17, 30000, 256001])
def test_many_nans_and_infinities(V, dtype):
    """Among the elements of one load too: the first NaN whatever stands before and after it."""
    g = torch.Generator().manual_seed(V)
    x = torch.randn(8, V + 7, generator=g).to(dtype)[:, :V]
    for row, share in enumerate((0.0, 1e-4, 0.01, 0.3, 1.0)):
        x[row, torch.rand(V, generator=g) < share] = float("nan")
    x[5:, torch.rand(V, generator=g) < 0.2] = float("inf")
    x[6, V // 2:] = float("nan")
    x[7] = -x[7]
    assert torch.equal(decode_ops.greedy_tokens(x.cuda()).cpu(), x.float().argmax(-1, keepdim=True).int())
