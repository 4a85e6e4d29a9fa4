"""Attention's forward against float64 at the edges of blocks and tiles, and of
the rule by which blocks find their head."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,B,H,G", [(64, 1, 3, 3), (128, 2, 8, 4),
                                     (64, 4, 8, 2), (128, 1, 5, 1)])
@pytest.mark.parametrize("S", [1, 31, 33, 64, 65, 127, 129, 192, 255, 256, 257, 320,
                               383, 512, 641])
@pytest.mark.parametrize("causal", [True, False])
def test_matches_float64(D, B, H, G, S, causal):
    from scaffold import ops

    torch.manual_seed(S + D)
    qkv = torch.randn(B, S, H + 2 * G, D, device="cuda").bfloat16()
    q, k, v = (t.transpose(1, 2) for t in qkv.split([H, G, G], 2))
    o, lse = ops.require_ext().attn_fwd(q, k, v, causal)
    kk, vv = (t.double().repeat_interleave(H // G, 1) for t in (k, v))
    s = q.double() @ kk.transpose(2, 3).contiguous() / math.sqrt(D)
    if causal:
        unseen = torch.ones(S, S, device="cuda", dtype=torch.bool).triu(1)
        s = s.masked_fill(unseen, -math.inf)
    w = torch.softmax(s, -1)
    # float32 scores of up to 8 deviations: 2^-20 of them
    assert (lse.double() - s.logsumexp(-1)).abs().max() < 2.0 ** -16
    # weights are rounded to 2^-9 of each (8 deviations of their sum over the
    # keys), the result to 2^-9 of it
    d = 8 * 2.0 ** -9 / math.sqrt(3) * ((w * w) @ (vv * vv)).sqrt()
    assert ((o.double() - w @ vv).abs() <= d + 2.0 ** -8 * (w @ vv).abs() + 2.0 ** -14).all()


def test_keys_that_lie_far_apart():
    """Rows 2^24 elements apart, as a view may have them."""
    from scaffold import ops

    torch.manual_seed(0)
    S, D = 70, 64
    wide = torch.empty(S, 1 << 24, device="cuda", dtype=torch.bfloat16)
    k = wide[:, :D].view(1, 1, S, D)
    k.copy_(torch.randn(1, 1, S, D, device="cuda"))
    q, v = (torch.randn(1, 1, S, D, device="cuda").bfloat16() for _ in range(2))
    f = ops.require_ext().prompt_attention
    assert torch.equal(f(q, k, v, S), f(q, k.contiguous(), v, S))
