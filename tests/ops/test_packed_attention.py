"""Attention of packed projections against attention of its three views, and
turned rows against rows that the vector kernel does not take."""

import pytest
import torch

from scaffold import ops


def _tables(S, D, dev):
    a = torch.outer(torch.arange(S, device=dev).float(),
                    10000.0 ** -(torch.arange(0, D, 2, device=dev) / D))
    return a.cos(), a.sin()


PLACES = [("cpu", torch.float32),
          pytest.param("cuda", torch.float32, marks=pytest.mark.gpu),
          pytest.param("cuda", torch.bfloat16, marks=pytest.mark.gpu)]


@pytest.mark.parametrize("dev,dt", PLACES, ids=str)
@pytest.mark.parametrize("B,S,H,G,D", [(1, 1, 1, 1, 64), (2, 70, 4, 2, 64),
                                       (3, 129, 8, 2, 128), (2, 33, 3, 3, 32),
                                       (1, 300, 12, 12, 64)])
@pytest.mark.parametrize("turn", [False, True])
def test_same_as_by_views(dev, dt, B, S, H, G, D, turn):
    torch.manual_seed(S)
    qkv = torch.randn(B, S, H + 2 * G, D, device=dev).to(dt).requires_grad_()
    do = torch.randn(B, S, H, D, device=dev).to(dt)
    cos, sin = _tables(S, D, dev) if turn else (None, None)
    got = ops.packed_attention(qkv, H, G, cos, sin)
    (dgot,) = torch.autograd.grad(got, qkv, do)
    q, k, v = (t.transpose(1, 2) for t in qkv.split([H, G, G], 2))
    if turn:
        q, k = ops.rope_apply(q, cos, sin), ops.rope_apply(k, cos, sin)
    want = ops.attention(q, k, v, causal=True).transpose(1, 2)
    (dwant,) = torch.autograd.grad(want, qkv, do)
    assert got.shape == do.shape and torch.equal(got, want)
    assert dgot.is_contiguous() and torch.equal(dgot, dwant)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,S,D", [(1, 1, 1, 8), (2, 5, 7, 64), (1, 40, 3, 128),
                                     (2, 3, 5, 24), (1, 2, 2, 2048)])
@pytest.mark.parametrize("inverse", [False, True])
def test_vectors_turn_as_pairs_do(B, H, S, D, inverse):
    f = ops.require_ext().rope_apply
    torch.manual_seed(D)
    cos, sin = _tables(S + 2, D, "cuda")
    odd = torch.randn(B, S, H, D + 1, device="cuda").bfloat16()[..., :D]
    odd = odd.transpose(1, 2)                  # rows of odd stride
    x = odd.transpose(1, 2).contiguous().transpose(1, 2)
    want = f(odd, cos, sin, inverse)
    assert torch.equal(f(x, cos, sin, inverse), want)
    room = torch.zeros(B, S, H + 3, D, device="cuda").bfloat16()
    place = room[:, :, 1:H + 1].transpose(1, 2)
    f(x, cos, sin, inverse, out=place)
    assert torch.equal(place, want)
    assert not room[:, :, 0].any() and not room[:, :, H + 1:].any()
    f(x, cos, sin, inverse, out=x)             # in place
    assert torch.equal(x, want)


@pytest.mark.gpu
@pytest.mark.parametrize("S", [(1 << 24) - 1, 1 << 24])
def test_turns_any_number_of_positions(S):
    """More positions than a launch has blocks of a position each."""
    f = ops.require_ext().rope_apply
    x = torch.randn(1, S, 4, 64, device="cuda", dtype=torch.bfloat16)
    cos = torch.full((S, 32), 0.6, device="cuda")
    sin = torch.full((S, 32), 0.8, device="cuda")
    x = x.transpose(1, 2)
    y = f(x, cos, sin, False)
    for part in (slice(0, 999), slice(S - 999, S)):
        t = x[:, :, part]
        assert torch.equal(y[:, :, part], f(t, cos[:999], sin[:999], False))
        u, w = t[..., ::2].float(), t[..., 1::2].float()
        got = y[:, :, part].float()
        # the result's rounding, half of 2^-8 of up to 1.4 times 6
        assert (got[..., ::2] - (0.6 * u - 0.8 * w)).abs().max() < 2 ** -5
        assert (got[..., 1::2] - (0.8 * u + 0.6 * w)).abs().max() < 2 ** -5


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,S,D", [
    (1, 31, 300, 8), (1, 32, 255, 8), (1, 32, 256, 8), (2, 11, 130, 24),
    (1, 40, 300, 128), (1, 1, 256, 256), (3, 2, 100, 2048), (1, 1, 256, 2056)])
@pytest.mark.parametrize("inverse", [False, True])
def test_vectors_turn_as_pairs_do_on_both_sides_of_the_rule(B, H, S, D, inverse):
    """Enough positions and elements for a block a position, and just not."""
    f = ops.require_ext().rope_apply
    torch.manual_seed(D)
    cos, sin = _tables(S, D, "cuda")
    odd = torch.randn(B, S, H, D + 1, device="cuda").bfloat16()[..., :D]
    odd = odd.transpose(1, 2)                  # rows of odd stride: by pairs
    x = odd.transpose(1, 2).contiguous().transpose(1, 2)
    want = f(odd, cos, sin, inverse)
    assert torch.equal(f(x, cos, sin, inverse), want)
    room = torch.zeros(B, S, H + 3, D, device="cuda").bfloat16()
    place = room[:, :, 1:H + 1].transpose(1, 2)
    f(x, cos, sin, inverse, out=place)
    assert torch.equal(place, want)
    assert not room[:, :, 0].any() and not room[:, :, H + 1:].any()
    f(x, cos, sin, inverse, out=x)             # in place
    assert torch.equal(x, want)
