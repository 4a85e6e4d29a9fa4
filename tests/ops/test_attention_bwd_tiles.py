"""Attention's backward at the edges of its blocks, tiles and masks, against
the same sums in float64."""

import pytest
import torch

from scaffold import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [31, 64, 127, 129, 255, 256, 257, 321, 383, 576])
@pytest.mark.parametrize("D,H,G", [(64, 2, 2), (64, 4, 1), (128, 2, 1), (128, 3, 3)])
@pytest.mark.parametrize("causal", [True, False])
def test_matches_float64(S, D, H, G, causal):
    torch.manual_seed(S + D)
    B = 2
    q, k, v, do = (torch.randn(B, n, S, D, device="cuda").bfloat16()
                   for n in (H, G, G, H))
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    o = ops.attention(*leaves, causal)
    dq, dk, dv = torch.autograd.grad(o, leaves, do)
    Q, K, V, dO = (t.double() for t in (q, k, v, do))
    K, V = (t.repeat_interleave(H // G, 1) for t in (K, V))
    s = Q @ K.transpose(2, 3) * D ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(S, S, device="cuda").triu(1).bool(), -torch.inf)
    P = torch.softmax(s, -1)
    O = P @ V
    delta = (dO * O).sum(-1, keepdim=True)
    dS = P * (dO @ V.transpose(2, 3) - delta) * D ** -0.5
    # P and dS enter the products in bf16 (2^-9 of each), and delta holds O's
    # rounding; everything is doubled for float32's share
    eP = 2.0 ** -8 * P
    eS = 2.0 ** -8 * (dS.abs() + P * (dO * O).abs().sum(-1, keepdim=True) * D ** -0.5)
    fold = lambda t: t.view(B, G, H // G, S, D).sum(2)
    T = lambda t: t.transpose(2, 3)
    for got, want, err in (
            (dq, dS @ K, eS @ K.abs()),
            (dk, fold(T(dS) @ Q), fold(T(eS) @ Q.abs())),
            (dv, fold(T(P) @ dO), fold(T(eP) @ dO.abs()))):
        assert ((got.double() - want).abs() <= err + 2.0 ** -8 * want.abs() + 1e-6).all()


@pytest.mark.parametrize("S", [64, 300])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("which", ["q", "k", "v", "do", "all"])
def test_operands_at_odd_places(S, D, which):
    """Rows of odd stride, and rows that start off 16 bytes, give what the same
    numbers in dense rows give."""
    torch.manual_seed(S + D)
    B, H, G = 2, 4, 2
    n = {"q": H, "k": G, "v": G, "do": H}
    dense = {a: torch.randn(B, n[a], S, D, device="cuda").bfloat16() for a in n}

    def run(t):
        leaves = [t[a].detach().requires_grad_() for a in "qkv"]
        o = ops.attention(*leaves, True)
        return o, *torch.autograd.grad(o, leaves, t["do"])

    want = run(dense)
    for pad, first in ((1, 0), (8, 3), (8, 8)):
        odd = dict(dense)
        for a in n if which == "all" else [which]:
            wide = torch.zeros(B, S, n[a], D + pad, device="cuda").bfloat16()
            odd[a] = wide[..., first:first + D].transpose(1, 2)
            odd[a].copy_(dense[a])
        for g, e in zip(run(odd), want):
            assert torch.equal(g, e)
