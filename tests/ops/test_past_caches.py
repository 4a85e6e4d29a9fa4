"""Passes whose operands and results are together more than the memory-side cache
holds, and go past it: batch norm of 64 MB, AdamW of 16 million elements."""

import pytest
import torch
import torch.nn.functional as F

from scaffold import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 64, 724, 725), (15, 2056, 33, 33)])
@pytest.mark.parametrize("relu", [True, False])
@pytest.mark.parametrize("use_res", [True, False])
def test_batch_norm(shape, relu, use_res):
    torch.manual_seed(1)
    N, C, H, W = shape
    assert N * C * H * W >= 1 << 25

    def image():
        return torch.randn(N, H, W, C, device="cuda").bfloat16().permute(0, 3, 1, 2)

    x, dy, res = image().requires_grad_(), image(), image() if use_res else None
    if use_res:
        res.requires_grad_()
    w = (torch.randn(C, device="cuda") * 0.1 + 1).requires_grad_()
    b = (torch.randn(C, device="cuda") * 0.1).requires_grad_()
    y = ops.batch_norm_act(x, res, w, b, torch.zeros(C, device="cuda"),
                           torch.ones(C, device="cuda"), 0.1, 1e-5, relu, True)
    ins = [t for t in (x, w, b, res) if t is not None]
    got = [y, *torch.autograd.grad(y, ins, dy)]
    ref = [t.detach().double().requires_grad_() for t in ins]
    z = F.batch_norm(ref[0], None, None, ref[1], ref[2], True, 0.1, 1e-5)
    z = z + ref[3] if use_res else z
    # the sign that passes is that of the float32 result
    z = z * (y > 0) if relu else z
    want = [z, *torch.autograd.grad(z, ref, dy.double())]
    for g, h in zip(got, want):
        assert (g.double() - h).norm() < 0.004 * h.norm()
        assert (g.double() - h).abs().max() < 0.05 * h.abs().max()


@pytest.mark.parametrize("sizes", [[(1 << 24) + 1], [1 << 24, 3, 4097, 1 << 20]])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_adamw(sizes, dtype):
    torch.manual_seed(2)
    p, m, g = ([torch.randn(s, device="cuda") for s in sizes] for _ in range(3))
    v = [torch.rand(s, device="cuda") for s in sizes]
    g = [t.to(dtype) for t in g]
    o = [torch.empty_like(t, dtype=torch.bfloat16) for t in p]
    kept = [[t.double() for t in ts] for ts in (p, m, v)]
    ops.fused_adamw_step(p, g, m, v, o, lr=1e-2, beta1=0.9, beta2=0.95, eps=1e-8,
                         weight_decay=0.1, step=3, grad_scale=0.5)
    for i in range(len(sizes)):
        gd = g[i].double() * 0.5
        rm = 0.9 * kept[1][i] + 0.1 * gd
        rv = 0.95 * kept[2][i] + 0.05 * gd * gd
        rp = kept[0][i] * (1 - 1e-3) - 1e-2 * (rm / (1 - 0.9 ** 3)) / (
            (rv / (1 - 0.95 ** 3)).sqrt() + 1e-8)
        for got, want in ((p[i], rp), (m[i], rm), (v[i], rv)):
            # a dozen roundings of 2^-24 of terms no larger than these
            assert ((got.double() - want).abs() <= 12 * 2.0 ** -24 * (want.abs() + 8)).all()
        assert torch.equal(o[i], p[i].bfloat16())
