"""The erf form of GELU: values, edges of vectors and of blocks."""

import pytest
import torch
import torch.nn.functional as F

from scaffold import ops

pytestmark = pytest.mark.gpu


def test_error_against_64_bits():
    z = torch.cat([torch.linspace(-12, 12, 1 << 20), torch.randn(1 << 20)]).cuda()
    want = F.gelu(z.double())
    err = (ops.gelu_erf(z).double() - want).abs()
    # the polynomial's 2e-8 of Phi and the roundings of 0.5, of the power and of the sum,
    # each 6e-8 of what it rounds
    assert (err <= 1e-7 * z.abs().clamp(min=0.5).double()).all()
    low = (z < -1) & (z > -6)
    assert (err[low] <= 3e-4 * want[low].abs()).all()


def test_ends():
    z = torch.tensor([torch.inf, -torch.inf, torch.nan, -1e30, 1e30, -17.0, 17.0, 0.0],
                     device="cuda")
    got, want = ops.gelu_erf(z), F.gelu(z.double()).float()
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 8, 2047, 2049, 8191, 1 << 22, (1 << 23) + 3])
@pytest.mark.parametrize("at", [0, 1])
def test_sizes(n, at, dtype):
    torch.manual_seed(n)
    z = torch.randn(n + at, device="cuda", dtype=dtype)[at:]
    want = F.gelu(z.double())
    got = ops.gelu_erf(z)
    half_ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    assert ((got.double() - want).abs() <= half_ulp * want.abs() + 1e-7 * z.abs().clamp(min=0.5)).all()
