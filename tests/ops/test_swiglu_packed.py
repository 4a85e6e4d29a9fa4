"""The packed SwiGLU against that of separate tensors, whose arithmetic is the
same to the bit, where blocks end inside rows and rows inside blocks."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,F", [
    (1, 8), (1, 2048), (257, 8), (85, 24), (3, 2056), (33, 2040), (300, 1792),
    (4097, 5632)])
def test_bits_of_separate_tensors(rows, F):
    from scaffold import ops

    torch.manual_seed(rows + F)
    gu = torch.randn(rows, 2 * F, device="cuda").bfloat16().requires_grad_()
    g, u = (t.detach().contiguous().requires_grad_() for t in gu.split(F, 1))
    dh = torch.randn(rows, F, device="cuda").bfloat16()
    want = ops.swiglu(g, u)
    got = ops.swiglu_packed(gu)
    assert torch.equal(got, want)
    dgu, = torch.autograd.grad(got, gu, dh)
    assert torch.equal(dgu, torch.cat(torch.autograd.grad(want, (g, u), dh), 1))
