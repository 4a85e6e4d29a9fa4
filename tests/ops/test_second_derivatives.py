"""Gradients of gradients through the linear ops on the GPU, against float64:
what a kernel without a gradient of its own would drop shows here."""

import pytest
import torch
import torch.nn.functional as F

from scaffold import ops

pytestmark = pytest.mark.gpu


def _penalty_grads(f, ins):
    """Gradients of the squared gradients of a sum of squares."""
    y = f(*ins)
    wide = torch.float64 if y.dtype == torch.float64 else torch.float32
    g = torch.autograd.grad(y.to(wide).square().sum(), ins, create_graph=True)
    return torch.autograd.grad(sum(t.to(wide).square().sum() for t in g), ins)


def _check(f, ref, ins):
    got = _penalty_grads(f, [t.clone().requires_grad_() for t in ins])
    want = _penalty_grads(ref, [t.double().requires_grad_() for t in ins])
    for g, e in zip(got, want):
        # about ten roundings of 2^-9 one behind the other, two of which are
        # squared; a dropped path is off by 0.13 and more
        assert (g.double() - e).norm() / e.norm() < 12 * 2.0 ** -9


def _operands(n):
    torch.manual_seed(n)
    x = torch.randn(37, 96, device="cuda").bfloat16()
    w = (torch.randn(n, 96, device="cuda") / 10).bfloat16()
    b = torch.randn(n, device="cuda").bfloat16()
    return x, w, b, torch.randn(37, n, device="cuda").bfloat16()


@pytest.mark.parametrize("n", [100, 200])
def test_linear(n):
    _check(ops.linear, F.linear, _operands(n)[:3])


@pytest.mark.parametrize("n", [100, 200])
def test_linear_residual(n):
    _check(ops.linear_residual, lambda x, w, b, r: F.linear(x, w, b) + r,
           _operands(n))


@pytest.mark.parametrize("n", [100, 200])
def test_linear_gelu(n):
    _check(ops.linear_gelu,
           lambda x, w, b: F.gelu(F.linear(x, w, b), approximate="tanh"),
           _operands(n)[:3])
