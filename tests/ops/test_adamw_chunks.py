"""AdamW over many tensors: chunks that lie in one tensor, across several, at odd
ends, and few elements."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [1 << 20, 4096, 4095, 1, 3, 4097, 1 << 18],          # chunks and ends
    [4097] * 300, [7] * 4096,                  # several to a chunk; few
    [5] * 3000 + [1 << 21] + [9] * 1000,                 # more than 64 times 64
    [(1 << 20) - 4], [1 << 20], [(1 << 20) + 1]])        # around the line between
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("out", [False, True])
def test_matches_float64(sizes, dtype, out):
    from scaffold import ops

    torch.manual_seed(len(sizes))
    total = sum((s + 3) // 4 * 4 for s in sizes)
    at = [0]
    for s in sizes:
        at.append(at[-1] + (s + 3) // 4 * 4)

    def split(t):
        return [t[a:a + s] for a, s in zip(at, sizes)]

    dev = "cuda"
    p, m = torch.randn(total, device=dev), 0.1 * torch.randn(total, device=dev)
    v, g = torch.rand(total, device=dev), torch.randn(total, device=dev).to(dtype)
    o = torch.full((total,), 7.0, device=dev, dtype=torch.bfloat16)
    keep = [t.clone() for t in (p, m, v)]
    lr, b1, b2, eps, wd, step, scale = 1e-2, 0.9, 0.95, 1e-8, 0.1, 3, 0.5
    ops.fused_adamw_step(split(p), split(g), split(m), split(v), split(o) if out else None,
                         lr=lr, beta1=b1, beta2=b2, eps=eps, weight_decay=wd, step=step,
                         grad_scale=scale)
    inside = torch.zeros(total, dtype=torch.bool, device=dev)
    for t in split(inside):
        t.fill_(True)
    rp, rm, rv = (t.double() for t in keep)
    gd = g.double() * scale
    rm = b1 * rm + (1 - b1) * gd
    rv = b2 * rv + (1 - b2) * gd * gd
    rp = rp * (1 - lr * wd) - lr * (rm / (1 - b1 ** step)) / ((rv / (1 - b2 ** step)).sqrt() + eps)
    # a dozen roundings of 2^-24 of terms no larger than these
    for got, want, before in ((p, rp, keep[0]), (m, rm, keep[1]), (v, rv, keep[2])):
        d = 12 * 2.0 ** -24 * (want.abs() + before.double().abs() + gd.abs().clamp(max=9) + 1)
        assert ((got.double() - want).abs() <= d)[inside].all()
        assert torch.equal(got[~inside], before[~inside])
    if out:
        assert torch.equal(o[inside], p.bfloat16()[inside])
        assert (o[~inside] == 7).all()
