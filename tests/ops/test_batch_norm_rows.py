"""batch_norm_act against float64 at the edges of its rules: rows that one
block keeps, rows that are streamed, ragged columns."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _exact(x, res, w, b, rm, rv, relu, dy):
    x, w, b, dy = (t.double() for t in (x, w, b, dy))
    x, w, b = (t.requires_grad_() for t in (x, w, b))
    res = None if res is None else res.double().requires_grad_()
    R = x.numel() / x.shape[1]

    def wide(t):
        return t.view(1, -1, 1, 1)

    mu = x.mean((0, 2, 3))
    var = (x - wide(mu)).square().mean((0, 2, 3))
    y = (x - wide(mu)) / torch.sqrt(wide(var) + 1e-5) * wide(w) + wide(b)
    y = y if res is None else y + res
    pre = y.detach()
    y = torch.relu(y) if relu else y
    ins = [x, w, b] + ([] if res is None else [res])
    g = torch.autograd.grad(y, ins, dy)
    ub = var * R / (R - 1) if R > 1 else var
    return (y.detach(), *g, (0.9 * rm.double() + 0.1 * mu).detach(),
            (0.9 * rv.double() + 0.1 * ub).detach()), pre


@pytest.mark.parametrize("N,C,H,W", [
    (1, 8, 1, 2), (2, 24, 3, 5), (1, 40, 5, 51), (1, 64, 1, 257),
    (32, 512, 7, 7), (2, 64, 32, 32), (1, 64, 1, 2049), (8, 24, 20, 20),
    (3, 2048, 7, 7), (4, 2056, 25, 25), (16, 128, 28, 28)])
@pytest.mark.parametrize("relu", [True, False])
@pytest.mark.parametrize("use_res", [True, False])
def test_matches_float64(N, C, H, W, relu, use_res):
    from scaffold import ops

    torch.manual_seed(N * C + W)

    def image(std=1.0, mean=0.0):
        t = torch.randn(N, H, W, C, device="cuda") * std + mean
        return t.bfloat16().permute(0, 3, 1, 2)

    x, dy = image(1.5, 0.2), image()
    res = image() if use_res else None
    w = torch.rand(C, device="cuda") + 0.5
    b = torch.randn(C, device="cuda") * 0.1
    rm, rv = torch.randn(C, device="cuda"), torch.rand(C, device="cuda") + 1
    want, pre = _exact(x, res, w, b, rm, rv, relu, dy)
    xs = x.clone().requires_grad_()
    rs = res.clone().requires_grad_() if use_res else None
    ws, bs = w.clone().requires_grad_(), b.clone().requires_grad_()
    y = ops.batch_norm_act(xs, rs, ws, bs, rm, rv, 0.1, 1e-5, relu, True)
    ins = [xs, ws, bs] + ([rs] if use_res else [])
    got = [y.detach(), *torch.autograd.grad(y, ins, dy), rm, rv]
    names = ["y", "dx", "dw", "db"] + (["dres"] if use_res else []) + ["rm", "rv"]
    # a pre-activation within float32's error of zero may pass or not: an
    # element (up to 4 of dy, 16 of dy * xhat) more or less in its channel's
    # sums, 1/R of which goes into every dx (times up to 1.5 / 1.4, and xhat)
    near = (pre.abs() < 1e-5) & relu
    flips = near.sum((0, 2, 3))
    R = x.numel() / C
    shift = (flips * (4 + 16 * 4) * 1.5 / R).view(1, -1, 1, 1)
    for name, g, e in zip(names, got, want):
        g, e = g.double(), e.double()
        if name in ("dw", "db"):
            bound = 1e-4 * R ** 0.5 + 16 * flips
            assert ((g - e).abs() <= bound + 1e-5 * e.abs()).all(), name
        elif name in ("rm", "rv"):
            assert torch.allclose(g, e, rtol=1e-5, atol=1e-5), name
        else:
            # one bf16 rounding (2^-9), float32 statistics behind it
            bound = 2.0 ** -8 * e.abs() + 1e-4 * e.abs().max()
            if name == "dx":
                bound = bound + shift
            ok = (g - e).abs() <= bound
            assert (ok | near).all(), (name, (g - e).abs().max())


@pytest.mark.parametrize("shape", [(0, 16, 7, 7), (3, 16, 0, 7)])
@pytest.mark.parametrize("relu", [True, False])
@pytest.mark.parametrize("use_res", [True, False])
def test_no_rows(shape, relu, use_res):
    """An empty batch, as the last one of an epoch can be: nothing is read, and
    the running statistics stay as on the CPU."""
    from scaffold import ops

    def image():
        return torch.randn(shape, device="cuda").bfloat16().requires_grad_()

    x, res = image(), image() if use_res else None
    w, b = (torch.rand(16, device="cuda").requires_grad_() for _ in range(2))
    rm, rv = torch.randn(16, device="cuda"), torch.rand(16, device="cuda")
    kept = rm.clone(), rv.clone()
    y = ops.batch_norm_act(x, res, w, b, rm, rv, 0.1, 1e-5, relu, True)
    assert y.shape == shape
    ins = [x, w, b] + ([res] if use_res else [])
    for t, g in zip(ins, torch.autograd.grad(y, ins, torch.ones_like(y))):
        assert g.shape == t.shape and not g.any()
    assert torch.equal(rm, kept[0]) and torch.equal(rv, kept[1])


@pytest.mark.parametrize("shape", [(2, 16, 4, 4), (2, 16, 33, 34)])
@pytest.mark.parametrize("use_res", [True, False])
def test_gradients_of_any_layout(shape, use_res):
    """What autograd hands back through cat (a slice of the channels), sum over
    the image (an expanded row) and slices of an image, all of stride(1) == 1,
    counts as the same numbers laid out like x."""
    from scaffold import ops

    torch.manual_seed(4)
    N, C, H, W = shape

    def image():
        t = torch.randn(N, H, W, C, device="cuda").bfloat16()
        return t.permute(0, 3, 1, 2).requires_grad_()

    x, res = image(), image() if use_res else None
    w, b = (torch.rand(C, device="cuda").requires_grad_() for _ in range(2))
    ins = [x, w, b] + ([res] if use_res else [])
    y = ops.batch_norm_act(x, res, w, b, torch.zeros(C, device="cuda"),
                           torch.ones(C, device="cuda"), 0.1, 1e-5, True, True)
    wide = torch.randn(N, H, W + 3, 3 * C, device="cuda").bfloat16()
    wide = wide.permute(0, 3, 1, 2)
    for dy in (wide[:, C:2 * C, :, 1:W + 1], wide[:, :C, :, :W],
               wide[:, :C, :1, :1].expand(shape), wide[:1, :C, :1, :1].expand(shape)):
        dense = dy.clone(memory_format=torch.channels_last)
        assert dy.stride(1) == 1 and dy.stride() != dense.stride()
        got = torch.autograd.grad(y, ins, dy, retain_graph=True)
        want = torch.autograd.grad(y, ins, dense, retain_graph=True)
        for g, e in zip(got, want):
            assert torch.equal(g, e)
    z = torch.cat([y, y.detach()], 1)
    assert torch.equal(torch.autograd.grad(z, x, wide[:, :2 * C, :, :W],
                                           retain_graph=True)[0],
                       torch.autograd.grad(y, x, wide[:, :C, :, :W],
                                           retain_graph=True)[0])
    rows = torch.randn(N, C, device="cuda").bfloat16()
    assert torch.equal(torch.autograd.grad(y.sum((2, 3)), x, rows, retain_graph=True)[0],
                       torch.autograd.grad(y, x, rows.view(N, C, 1, 1).repeat(
                           1, 1, H, W))[0])


def test_refuses_operands_that_do_not_fit():
    """Sizes that the kernels would read past: refused on the host."""
    from scaffold import ops

    C = 16
    x = torch.randn(2, C, 5, 5, device="cuda").bfloat16()
    vec = {n: torch.ones(C, device="cuda") for n in ("w", "b", "m", "v")}

    def call(x=x, res=None, **kw):
        p = {**vec, **kw}
        return ops.batch_norm_act(x, res, p["w"], p["b"], p["m"], p["v"], 0.1,
                                  1e-5, True, True)

    call()
    for n in "wbmv":
        for bad in (torch.ones(C - 8, device="cuda"), torch.ones(C),
                    torch.ones(2 * C, device="cuda")[::2]):
            with pytest.raises(RuntimeError):
                call(**{n: bad})
    with pytest.raises(RuntimeError):
        call(m=None)
    for bad in (x[:1], x[:, :8], x[..., :4], x.float()):
        with pytest.raises(RuntimeError):
            call(res=bad)
    with pytest.raises(RuntimeError):
        call(x=x[:, :0], **{n: t[:0] for n, t in vec.items()})
    ext, nhwc = ops.require_ext(), torch.channels_last
    x = x.contiguous(memory_format=nhwc)
    y, mean, rstd = ext.bn_fwd(x, None, vec["w"], vec["b"], None, None, 0.1,
                               1e-5, True)
    ext.bn_bwd(y, x, False, None, vec["w"], vec["b"], mean, rstd, True)
    for dy, xx in ((y[:1], x), (y.float(), x), (y, x.contiguous()),
                   (y[:, :, 1:], x[:, :, 1:])):
        with pytest.raises(RuntimeError):
            ext.bn_bwd(dy, xx, False, None, vec["w"], vec["b"], mean, rstd, True)


def test_benchmark_runs():
    """benchmarks/bn_only.py calls the kernels as they are."""
    import runpy
    from pathlib import Path

    runpy.run_path(str(Path(__file__).parents[2] / "benchmarks" / "bn_only.py"))


@pytest.mark.parametrize("R", [4 * 65535, 4 * 65535 + 1, 300001])
def test_more_rows_than_a_grid_of_four(R):
    """Rows of 2048 channels, four to a block, up to and beyond a grid's limit;
    channels are independent, so that eight of them tell."""
    from scaffold import ops

    torch.manual_seed(R)
    C = 2048
    x, dy, res = (torch.randn(1, R, 1, C, device="cuda", dtype=torch.bfloat16)
                  .permute(0, 3, 1, 2) for _ in range(3))
    w, b = torch.rand(C, device="cuda") + 0.5, torch.randn(C, device="cuda") * 0.1
    rm, rv = torch.zeros(C, device="cuda"), torch.ones(C, device="cuda")
    some = [0, 7, 8, 1023, 1024, 2039, 2040, 2047]
    want, pre = _exact(*(t[:, some] for t in (x, res)),
                       *(t[some] for t in (w, b, rm, rv)), True, dy[:, some])
    ins = [t.requires_grad_() for t in (x, w, b, res)]
    y = ops.batch_norm_act(x, res, w, b, rm, rv, 0.1, 1e-5, True, True)
    dx, _, _, dres = torch.autograd.grad(y, ins, dy)
    for name, g, e in (("y", y, want[0]), ("dx", dx, want[1]), ("dres", dres, want[4])):
        # one bf16 rounding (2^-9), float32 statistics behind it; a sign within
        # float32's error of zero may fall on either side
        g = g.detach()[:, some].double()
        bound = 2.0 ** -8 * e.abs() + 1e-4 * e.abs().max()
        assert (((g - e).abs() <= bound) | (pre.abs() < 1e-5)).all(), name
