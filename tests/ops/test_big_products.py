"""Large products by tiles: at the edges of tiles, over several tiles a block,
past the caches."""

import warnings

import pytest
import torch
import torch.nn.functional as F

from scaffold import ops

pytestmark = pytest.mark.gpu


def _close(got, a, b):
    """got = a b, of which every partial sum is below the sum of sizes: the
    result's rounding, and that of depth / 32 + 32 float32 sums."""
    a, b = a.double(), b.double()
    want, size = a @ b, a.abs() @ b.abs()
    lim = 2.0 ** -8 * want.abs() + (a.shape[1] / 32 + 32) * 2.0 ** -24 * size
    assert got.shape == want.shape and ((got.double() - want).abs() <= lim).all()


def _rows(n, m, mean=0.0):
    """n rows of m, and NaN behind the last"""
    t = torch.full((n + 64, m), torch.nan, device="cuda").bfloat16()
    t[:n] = torch.randn(n, m, device="cuda") + mean
    return t[:n]


@pytest.mark.parametrize("T,N,K", [
    (257, 5128, 8200),        # three tiles a block, the last ones partly empty
    (4097, 3080, 3600),       # one tile a block, the last ones of eight rows
    (300, 8192, 7432),        # a result that goes past the caches
    (385, 10000, 1280)])
def test_weight_gradients(T, N, K):
    torch.manual_seed(T)
    dy, x = _rows(T, N), _rows(T, K, 0.5)
    got = ops.require_ext().wide_weight_grad(dy, x)
    _close(got, dy.t(), x)
    assert torch.equal(got, ops.require_ext().wide_weight_grad(dy, x))


def test_weight_gradients_of_other_operands_are_left():
    f = ops.require_ext().wide_weight_grad
    dy, x = _rows(2048, 3328), _rows(2048, 3584)
    assert f(dy, x) is not None
    for a, b in ((dy.half(), x.half()), (dy, x[:-1]), (dy[:, :-4], x),
                 (dy.t().contiguous().t(), x), (dy.cpu(), x), (dy[:128], x[:128]),
                 (dy.clone().requires_grad_(), x)):
        assert f(a, b) is None


def test_infinite_rows_stay_where_they_are():
    torch.manual_seed(3)
    dy, x = _rows(2048, 3328), _rows(2048, 3584)
    dy[:, 300] = torch.inf
    got = ops.require_ext().wide_weight_grad(dy, x)
    assert not got[300].isfinite().any()
    rest = torch.cat([got[:300], got[301:]])
    _close(rest, torch.cat([dy[:, :300], dy[:, 301:]], 1).t(), x)


@pytest.mark.parametrize("M,N,K", [
    (505, 128, 32760),        # one stage of each half, edges both ways
    (5003, 256, 2568),        # tiles of 256 columns, the last of eight
    (16001, 384, 760),        # of 192, one of them of one row
    (16000, 2304, 760),
    (8192, 640, 7432)])       # past the caches
def test_input_gradients(M, N, K):
    torch.manual_seed(M)
    dy = _rows(M, N)
    w = _rows(N, K, 0.5)
    got = ops.require_ext().input_grad(dy, w)
    _close(got, dy, w)
    assert torch.equal(got, ops.require_ext().input_grad(dy, w))


def test_input_gradients_of_other_operands_are_left():
    f = ops.require_ext().input_grad
    dy, w = _rows(4096, 512), _rows(512, 4096)
    assert f(dy, w) is not None
    for a, b in ((dy.half(), w.half()), (dy[:, :-8], w), (dy, w.t()),
                 (dy[:, :448].contiguous(), w[:448].contiguous()), (dy.cpu(), w),
                 (dy[:128], w), (dy, w.clone().requires_grad_())):
        assert f(a, b) is None


@pytest.mark.parametrize("act", [False, True])
def test_layers_take_it(act, monkeypatch):
    ext, calls = ops.require_ext(), []
    made = ext.input_grad
    monkeypatch.setattr(ext, "input_grad",
                        lambda *a: calls.append(1) or made(*a))
    torch.manual_seed(1)
    x = torch.randn(4096, 4096, device="cuda").bfloat16().requires_grad_()
    w = (torch.randn(512, 4096, device="cuda") / 64).bfloat16().requires_grad_()
    b = torch.zeros(512, device="cuda").bfloat16().requires_grad_()
    y = (ops.linear_gelu if act else ops.linear)(x, w, b)
    dy = torch.randn_like(y)
    (dx,) = torch.autograd.grad(y, x, dy, retain_graph=True)
    assert len(calls) == 1
    if not act:
        _close(dx, dy, w.detach())
    torch.autograd.grad(y, x, dy.requires_grad_(), create_graph=True)
    assert len(calls) == 1


@pytest.mark.parametrize("M,N,K", [(300, 15001, 768), (255, 4096, 4096), (20000, 1000, 12),
                                   (64, 264, 160000), (13000, 264, 768)])
def test_sizes_that_are_no_kernel_s_are_not_asked_about(M, N, K, monkeypatch):
    ext, calls = ops.require_ext(), []
    for name in ("input_grad", "wide_weight_grad"):
        monkeypatch.setattr(ext, name, lambda *a: calls.append(1))
    x, w = _rows(M, K).requires_grad_(), (_rows(N, K) / K ** 0.5).requires_grad_()
    y = ops.linear(x, w)
    dy = torch.randn_like(y)
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    assert not calls
    assert dx.shape == x.shape and dw.shape == w.shape


@pytest.mark.parametrize("M,N,K,act,bias", [
    (16129, 2056, 256, 0, True),      # tiles of 256 columns, several a block
    (16001, 768, 768, 0, True),       # of 192, the last of one row
    (2500, 8184, 1408, 0, False),     # of 192, the last of 120 columns
    (9000, 6664, 256, 0, False),      # past the caches
    (4100, 5128, 1152, 2, False),
    (16001, 768, 768, 2, True),
    (2040, 8192, 2048, 2, False)])
def test_products(M, N, K, act, bias):
    torch.manual_seed(M)
    x, w = _rows(M, K), _rows(N, K, 0.5) / K ** 0.5
    b = torch.randn(N, device="cuda").bfloat16() if bias else None
    got = ops.require_ext().tile_linear(x, w.contiguous(), b, act)
    a, v = x.double(), w.double().t()
    size = a.abs() @ v.abs() + (b.double().abs() if bias else 0)
    want = a @ v + (b.double() if bias else 0)
    lim = (K / 32 + 34) * 2.0 ** -24 * size
    if act:                           # whose slope is below 1.13
        want, lim = F.gelu(want), 1.13 * lim + 1e-7 * want.abs().clamp(min=0.5)
    assert ((got.double() - want).abs() <= lim + 2.0 ** -8 * want.abs()).all()


@pytest.mark.parametrize("M,N,K,act,own", [
    (10000, 2176, 1024, 0, True), (10000, 2176, 1152, 0, False),    # 0.65 of two rounds
    (7000, 1792, 512, 0, True), (7000, 1792, 640, 0, False),        # whole across, one
    (7000, 1920, 640, 0, True),
    (6500, 4096, 1280, 0, True), (6500, 4096, 1408, 0, False),      # whole across, two
    (6500, 4096, 2048, 0, False), (6500, 4096, 2176, 0, True),
    (2456, 15360, 2048, 2, True), (2456, 15360, 2176, 2, False),    # 0.75 of three
    (2456, 15368, 2176, 2, True)])
def test_whole_tiles_of_part_of_a_round(M, N, K, act, own):
    """Where a library is as quick; both ways are one rounding of the same sums."""
    torch.manual_seed(M)
    x, w = _rows(M, K), (_rows(N, K, 0.5) / K ** 0.5).contiguous()
    assert (ops.require_ext().tile_linear(x, w, None, act) is not None) == own
    if act == 0:
        with torch.no_grad():
            _close(ops.linear(x, w), x, w.t())


def test_rows_that_lie_far_apart():
    torch.manual_seed(5)
    both = _rows(8000, 1024)
    w = _rows(2048, 512)
    got = ops.require_ext().tile_linear(both[:, 512:], w)
    _close(got, both[:, 512:], w.t())


@pytest.mark.parametrize("M,N,K,bias", [
    (16001, 768, 768, True),          # 192 columns, the last tile of one row
    (2500, 8184, 1408, False),        # the last of 120 columns
    (16384, 768, 768, True),
    (16129, 2056, 256, True),         # 256 columns, several tiles a block
    (9000, 6664, 256, False)])        # past the caches
def test_products_beside_a_residual(M, N, K, bias):
    torch.manual_seed(M)
    x, w, res = _rows(M, K), (_rows(N, K, 0.5) / K ** 0.5).contiguous(), _rows(M, N)
    b = torch.randn(N, device="cuda").bfloat16() if bias else None
    got = ops.require_ext().residual_linear(x, w, b, res, False)
    # the residual and the bias are two more terms of each sum
    want = x.double() @ w.double().t() + res.double() + (b.double() if bias else 0)
    size = x.double().abs() @ w.double().abs().t() + res.double().abs() + (
        b.double().abs() if bias else 0)
    lim = 2.0 ** -8 * want.abs() + (K / 32 + 34) * 2.0 ** -24 * size
    assert ((got.double() - want).abs() <= lim).all()
    apart = ops.require_ext().tile_linear(x, w, b, 0) + res
    assert torch.equal(ops.require_ext().residual_linear(x, w, b, res, True), apart)
    if M % 128 == 0 and N % 128 == 0:
        assert torch.equal(got, ops.require_ext().linear_fwd(x, w, b, 2, res)[0])


def test_residuals_of_other_forms_are_left():
    def f(*a):
        return ops.require_ext().residual_linear(*a, False)

    x, w, b, r = _rows(16384, 768), _rows(768, 768), _rows(1, 768)[0], _rows(16384, 768)
    assert f(x, w, b, r) is not None and f(x.view(4, 4096, 768), w, b, r.view(4, 4096, 768)) is not None
    odd = torch.cat([r[0, :1], r.flatten()])[1:].view_as(r)
    for other in (r[:1], r[:, :1], r.float(), odd, r.cpu(), r.t().contiguous().t(),
                  r.view(4, 4096, 768)):
        assert f(x, w, b, other) is None


@pytest.mark.parametrize("n", [768, 3072])
def test_residual_layers_take_it(n, monkeypatch):
    """Both layers that add a residual, and their gradients; a residual that is
    spread over rows is added as before."""
    ext, calls = ops.require_ext(), []
    made = ext.residual_linear
    monkeypatch.setattr(ext, "residual_linear",
                        lambda *a: calls.append(made(*a)) or calls[-1])
    torch.manual_seed(n)
    x, r = (torch.randn(16384, k, device="cuda").bfloat16().requires_grad_() for k in (n, 768))
    w = (torch.randn(768, n, device="cuda") / n ** 0.5).bfloat16().requires_grad_()
    b = torch.randn(768, device="cuda").bfloat16().requires_grad_()
    y = ops.linear_residual(x, w, b, r)
    assert len(calls) == 1 and calls[0] is not None
    dy = torch.randn_like(y)
    got = torch.autograd.grad(y, (x, w, b, r), dy)
    want = torch.autograd.grad(ops.linear(x, w, b), (x, w, b), dy)
    assert all(map(torch.equal, got, (*want, dy)))
    if n == 3072:
        y = ops.linear_residual(x, w, b, r[:1])
        assert torch.equal(y, ops.linear(x, w, b) + r[:1])
        (got,) = torch.autograd.grad(y, r, dy)
        assert got.shape == r.shape and not got[1:].any()


@pytest.mark.parametrize("M,N,K,own", [
    # nothing, also where one is large enough to be asked about
    (100, 1024, 2816, False), (3200, 1408, 1664, False), (4682, 2048, 1024, False),
    (721, 3072, 5632, False), (255, 4096, 14336, False), (4096, 2056, 128, False),
    # the product, by tiles
    (500, 2048, 2048, True),
    # a gradient alone, of less and of more than 10 G products
    (408, 2048, 5632, False), (1800, 2048, 5632, True), (7015, 768, 1536, False),
    (6628, 512, 3536, True),
    # a weight gradient of few tiles, out of few and many rows
    (8192, 256, 1032, False), (22184, 456, 480, True), (32767, 72, 104, False),
    (32768, 72, 104, True), (40000, 56, 104, False)])
def test_residuals_without_a_bias_are_torch_s_where_nothing_is_ours(M, N, K, own):
    x = torch.randn(M, K, device="cuda").bfloat16().requires_grad_()
    w = (torch.randn(N, K, device="cuda") / K ** 0.5).bfloat16().requires_grad_()
    res = torch.randn(M, N, device="cuda").bfloat16()
    y = ops.linear_residual(x, w, None, res)
    assert (type(y.grad_fn).__name__ == "_LinearLibBackward") == own
    # two roundings, of which the first may differ
    torch.testing.assert_close(y, F.linear(x, w) + res, rtol=2 ** -7, atol=2 ** -6)


class Marked(torch.Tensor):
    pass


@pytest.mark.filterwarnings("ignore:.*torch.jit.trace:DeprecationWarning",
                            "ignore::torch.jit.TracerWarning")
def test_residuals_without_a_bias_that_torch_has_to_see():
    x = torch.randn(4096, 768, device="cuda").bfloat16().requires_grad_()
    w = (torch.randn(3072, 768, device="cuda") / 28).bfloat16().requires_grad_()
    res = torch.randn(4096, 3072, device="cuda").bfloat16()
    f = ops.linear_residual
    assert type(f(x, w, None, res).grad_fn).__name__ == "_LinearLibBackward"
    assert type(f(x, w, None, res.as_subclass(Marked)).grad_fn).__name__ != "_LinearLibBackward"
    traced = torch.jit.trace(lambda x, w, r: f(x, w, None, r), (x, w, res), check_trace=False)
    assert "PythonOp" not in str(traced.graph) and "_LinearLib" not in str(traced.graph)
    # a weight of one row without its dimension
    x = torch.randn(4096, 2048, device="cuda").bfloat16()
    v = torch.randn(2048, device="cuda").bfloat16().requires_grad_()
    (got,) = torch.autograd.grad(f(x, v, None, res[:, 0]).sum(), v)
    assert got.shape == v.shape


def test_deep_products_of_training_stay_with_the_library():
    """What a gradient goes through does; without one the kernel of tiles is as good."""
    torch.manual_seed(0)
    x, w = _rows(1000, 4096), (_rows(28672, 4096) / 64).contiguous()
    f = ops.require_ext().tile_linear
    assert f(x, w, None, 0, True) is None
    _close(f(x, w), x, w.t())
    _close(ops.linear(x.clone().requires_grad_(), w).detach(), x, w.t())
    x, w, res = _rows(3000, 4096), (_rows(4096, 4096) / 64).contiguous(), _rows(3000, 4096)
    assert ops.require_ext().residual_linear(x, w, None, res, True) is None


@pytest.mark.parametrize("T,own", [(4096, True), (5000, True), (6002, False), (8192, True)])
def test_deep_gradients(T, own):
    """Those of part of a round of tiles stay with the library; the others are right,
    whether or not they are its bits."""
    ext = ops.require_ext()
    torch.manual_seed(T)
    w, x, dy = _rows(4096, 14336).contiguous(), _rows(T, 14336), _rows(T, 4096)
    dx, dw = ext.input_grad(dy, w), ext.wide_weight_grad(dy, x)
    assert (dx is not None) == own and (dw is not None) == (T == 4096)
    same = []
    if own:
        _close(dx, dy, w)
        same.append(("dx", torch.equal(dx, dy @ w)))
    if T == 4096:
        _close(dw, dy.t(), x)
        same.append(("dw", torch.equal(dw, dy.t() @ x)))
    # in the bits of the library that the rules were made for; another may sum otherwise
    if not all(s for _, s in same):
        warnings.warn(f"the library sums in another order: {same}")
