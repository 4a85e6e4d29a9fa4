"""Gradients that are not the bucket's own views come into it as they are."""

import pytest
import torch
import torch.nn as nn

from scaffold.dist.ddp import BucketedDDP

PLACES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


def _step(dev, change):
    """Gradients in the bucket after a backward, change(params), finish()."""
    torch.manual_seed(0)
    net = nn.Sequential(nn.Linear(6, 6), nn.Linear(6, 3)).to(dev)
    ddp = BucketedDDP(net)
    ddp.zero_grad()
    with ddp.no_sync():                  # .grad are the views afterwards
        ddp(torch.ones(4, 6, device=dev)).square().sum().backward()
    change(list(net.parameters()))
    ddp.finish()
    for b in ddp.buckets:
        assert all(p.grad is v for p, v in zip(b.params, b.views))
    return [p.grad.clone() for p in net.parameters()]


def _replace(f):
    def change(params):
        for p in params:
            p.grad = f(p.grad)
    return change


@pytest.mark.parametrize("dev", PLACES)
def test_replaced_by_the_same_numbers(dev):
    want = _step(dev, lambda params: None)
    assert all(g.any() for g in want)
    for f in (torch.Tensor.detach, torch.clone, lambda g: g.view_as(g),
              lambda g: g.t().contiguous().t() if g.dim() == 2 else g):
        for g, w in zip(_step(dev, _replace(f)), want):
            assert torch.equal(g, w)


@pytest.mark.parametrize("dev", PLACES)
def test_replaced_by_others(dev):
    want = _step(dev, lambda params: None)
    for g, w in zip(_step(dev, _replace(lambda g: 2 * g)), want):
        assert torch.equal(g, 2 * w)
    for g in _step(dev, _replace(lambda g: None)):
        assert not g.any()

    def turn(params):                    # in the bucket, laid out otherwise
        params[0].grad = params[0].grad.t()

    got = _step(dev, turn)
    assert torch.equal(got[0], want[0].t()) and torch.equal(got[2], want[2])


@pytest.mark.parametrize("dev", PLACES)
def test_sparse_ones(dev):
    """Also into views that do not start where the bucket does."""
    want = _step(dev, lambda params: None)
    for g, w in zip(_step(dev, _replace(lambda g: g.to_sparse())), want):
        assert torch.equal(g, w)
