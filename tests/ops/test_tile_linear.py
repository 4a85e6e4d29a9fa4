"""Products of some hundred rows by tiles, at the edges of tiles, of stages and of
what takes which tile."""

import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


# tiles of 64 x 64 up to 256 of them, 128 x 64, 128 x 128, 128 x 256; depths of
# one stage, of fewer than lie in LDS and of no whole round of them
@pytest.mark.parametrize("M,N,K", [
    (96, 2048, 64), (97, 1000, 128), (127, 1544, 192), (129, 5000, 320),
    (1024, 1024, 576), (1025, 1024, 64), (1000, 2056, 704), (2047, 1032, 128),
    (2048, 2040, 64), (1153, 3072, 192), (1920, 2048, 448), (2049, 2816, 64),
    (2300, 2560, 128), (4096, 3000, 320), (1665, 2040, 2112), (641, 4600, 4160)])
@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("bias", [False, True])
def test_matches_float64(M, N, K, act, bias):
    from scaffold import ops

    torch.manual_seed(M + N + K)
    dev = "cuda"
    x = torch.randn(M, K + 8, device=dev).bfloat16()
    x[:, K:] = float("nan")
    x = x[:, :K]
    w = (torch.randn(N, K, device=dev) / math.sqrt(K)).bfloat16()
    b = torch.randn(N, device=dev).bfloat16() if bias else None
    got = ops.require_ext().tile_linear(x, w, b, act)
    if got is None:                  # the widest tile with nothing behind it
        assert act == 0 and -(-M // 128) * -(-N // 128) > 256
        return
    y = x.double() @ w.double().T
    if bias:
        y = y + b.double()
    if act:
        y = F.gelu(y, approximate="tanh" if act == 1 else "none")
    # one rounding of the result (2^-9 of it); sums of K products and the
    # exponential in float32 are far below
    assert ((got.double() - y).abs() <= 2.0 ** -8 * y.abs() + 2.0 ** -14).all()


def test_infinite_weights_stay_where_they_are():
    from scaffold import ops

    x = torch.ones(200, 448, device="cuda", dtype=torch.bfloat16)
    w = torch.ones(1024, 448, device="cuda", dtype=torch.bfloat16)
    w[5, -1] = float("inf")
    got = ops.require_ext().tile_linear(x, w)
    assert (got[:, 5] == float("inf")).all()
    got[:, 5] = 0
    assert got.isfinite().all()


def test_leaves_what_it_is_not_for():
    from scaffold import ops

    f = ops.require_ext().tile_linear
    x = torch.randn(200, 512, device="cuda").bfloat16()
    w = torch.randn(1024, 512, device="cuda").bfloat16()
    assert f(x, w) is not None and f(x.view(2, 100, 512), w).shape == (2, 100, 1024)
    assert f(x[:64], w) is None                    # few rows
    assert f(x[:, :96], w[:, :96].contiguous()) is None       # depth
    assert f(x[:, 4:68], w[:, :64].contiguous()) is None      # alignment
    assert f(x, w[:1020]) is None                  # columns in eights
    assert f(x.float(), w.float()) is None and f(x, w.float()) is None
    assert f(x[:1].expand(200, 512), w) is None    # rows in one place
    assert f(x, w.requires_grad_()) is None        # a graph is wanted
    with torch.no_grad():
        assert f(x, w) is not None
        assert torch.func.vmap(lambda v: F.linear(v, w))(x.view(2, 100, 512)).shape == (2, 100, 1024)
    y = ops.linear(x.requires_grad_(), w)
    gx, gw = torch.autograd.grad(y.float().square().sum(), [x, w])
    rx, rw = torch.autograd.grad(F.linear(x.double(), w.double()).square().sum(), [x, w])
    for g, r in ((gx, rx), (gw, rw)):
        # y rounded, and the gradient of it, and the result: 2^-9 each
        assert (g.double() - r.double()).norm() <= 3 * 2.0 ** -9 * r.double().norm()


@pytest.mark.parametrize("grad", [False, True])
def test_seen_by_modes_and_by_the_compiler(grad):
    """A product stays a product for what counts or traces calls."""
    from torch.utils.flop_counter import FlopCounterMode

    from scaffold import ops

    x, w = (torch.randn(n, 768, device="cuda").bfloat16() for n in (256, 2304))
    with torch.set_grad_enabled(grad):
        with FlopCounterMode(display=False) as flops:
            y = ops.linear(x, w)
        assert flops.get_total_flops() == 2 * 256 * 768 * 2304
        whole = torch.compile(lambda t: ops.linear(t, w), backend="eager", fullgraph=True)
        # one rounding either way
        torch.testing.assert_close(whole(x), y, rtol=2 ** -7, atol=2 ** -10)
