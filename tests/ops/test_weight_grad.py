"""Weight gradients out of many rows, at the edges of tiles, stages and parts."""

import pytest
import torch

from scaffold import ops

pytestmark = pytest.mark.gpu


def _close(got, dy, x):
    want = dy.double().T @ x.double()
    # the result's rounding, and sums of T products in float32: every partial
    # sum is below the sum of sizes, T / 64 + 64 roundings deep
    size = dy.double().abs().T @ x.double().abs()
    lim = 2.0 ** -8 * want.abs() + (len(x) / 32 + 64) * 2.0 ** -24 * size
    assert ((got.double() - want).abs() <= lim).all()


@pytest.mark.parametrize("N,K", [(8, 8), (256, 256), (264, 248), (520, 1016),
                                 (768, 768), (4096, 1024)])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 127, 129, 1000, 8192, 8225])
def test_matches_float64(N, K, T):
    torch.manual_seed(N + K + T)
    dy = torch.randn(T, N, device="cuda").bfloat16()
    x = (torch.randn(T, K, device="cuda") + 0.5).bfloat16()
    # what lies behind the last row must not count
    rows = torch.full((T + 64, N), torch.nan, device="cuda").bfloat16()
    rows[:T] = dy
    got = ops.require_ext().weight_grad(rows[:T], x)
    _close(got, dy, x)
    assert torch.equal(got, ops.require_ext().weight_grad(dy, x))


@pytest.mark.parametrize("T,N,K,own", [
    (8192, 64, 72, True), (8191, 64, 72, False), (8192, 64, 68, False),
    (8192, 4096, 1032, False), (8192, 4096, 1024, True)])
@pytest.mark.parametrize("act", [False, True])
def test_layers_take_it(T, N, K, own, act, monkeypatch):
    torch.manual_seed(1)
    ext, calls = ops.require_ext(), []
    made = ext.weight_grad
    monkeypatch.setattr(ext, "weight_grad",
                        lambda *a: calls.append(1) or made(*a))
    x = torch.randn(T, K, device="cuda").bfloat16().requires_grad_()
    w = (torch.randn(N, K, device="cuda") / K ** 0.5).bfloat16().requires_grad_()
    b = torch.zeros(N, device="cuda").bfloat16().requires_grad_()
    y = (ops.linear_gelu if act else ops.linear)(x, w, b)
    dy = torch.randn_like(y)
    (dw,) = torch.autograd.grad(y, w, dy, retain_graph=True)
    assert len(calls) == own
    if not act:
        _close(dw, dy, x.detach())
    # a graph of the backward stays with operations that have one (what such a
    # graph yields: test_second_derivatives.py): dw is linear in dy
    (dw2,) = torch.autograd.grad(y, w, dy.requires_grad_(), create_graph=True)
    (back,) = torch.autograd.grad(dw2, dy, torch.ones_like(dw2))
    assert len(calls) == own and back.any(0).all()


def test_refuses_other_operands():
    f = ops.require_ext().weight_grad
    a = torch.zeros(64, 16, device="cuda", dtype=torch.bfloat16)
    for dy, x in ((a, a[:32]), (a, a.float()), (a[:, :12].contiguous(), a),
                  (a.t(), a.t()), (a[:0], a[:0]), (a[:, 0], a)):
        with pytest.raises(RuntimeError):
            f(dy, x)


@pytest.mark.parametrize("N,K,own", [
    (56, 4096, False), (4096, 56, False), (64, 8192, True), (64, 8200, False),
    (248, 16384, False), (256, 16384, True), (8, 8, False)])
def test_tiles_that_are_mostly_empty_stay_with_the_library(N, K, own, monkeypatch):
    ext, calls = ops.require_ext(), []
    made = ext.weight_grad
    monkeypatch.setattr(ext, "weight_grad",
                        lambda *a: calls.append(1) or made(*a))
    torch.manual_seed(N)
    dy = torch.randn(8192, N, device="cuda").bfloat16()
    x = torch.randn(8192, K, device="cuda").bfloat16()
    with torch.no_grad():
        _close(ops._weight_grad(dy, x), dy, x)
    assert len(calls) == own
