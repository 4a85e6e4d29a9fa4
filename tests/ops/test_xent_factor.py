"""The factor of cross-entropy's gradient, the loss's own over the rows, is
rounded once."""

import numpy as np
import pytest
import torch

from scaffold import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 3, 7, 11, 33, 100, 999, 16384])
@pytest.mark.parametrize("d", [1.0, 0.3, 7.77, 1e-3, 65536.0, 3.0e38])
def test_rounded_once(R, d):
    # a target of no probability: its gradient is the factor and nothing else
    x = torch.zeros(R, 3, device="cuda")
    x[:, 1] = -1e4
    x.requires_grad_()
    loss = ops.softmax_cross_entropy(
        x, torch.ones(R, dtype=torch.int64, device="cuda"))
    d = torch.tensor(d, device="cuda")
    (dx,) = torch.autograd.grad(loss, x, d)
    want = -np.float32(np.float64(d.item()) / R)
    assert (dx[:, 1] == want.item()).all()
