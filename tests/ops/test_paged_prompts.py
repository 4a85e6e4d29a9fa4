"""Attention over pages, in portions and single tokens that end at the edges of
waves, tiles and pages, for head sizes that fill their images and ones that do
not."""

import math

import pytest
import torch

from tests.oracle import lasezen as L
from tests.oracle.places import close, rnd
from tests.unit.test_lasezen_ops import run_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,d,e", [(4, 2, 128, 128), (3, 3, 64, 128), (6, 2, 128, 64),
                                     (8, 2, 64, 64), (2, 1, 72, 40), (5, 1, 104, 128)])
@pytest.mark.parametrize("parts,size,sink", [
    ((33,), 0, True), ((64, 65), 48, False), ((97, 2, 63), 129, True),
    ((31, 128, 40), 0, False), ((30, 1, 1, 1, 30, 1, 1, 1), 48, True),
    ((127, 1, 1), 129, False), ((300, 1, 1), 0, True)], ids=str)
def test_matches_oracle(H, G, d, e, parts, size, sink):
    T = sum(parts)
    q, k, v = rnd(T, H, d, seed=1), rnd(T, G, d, seed=2), rnd(T, G, e, seed=3)
    s = rnd(H, seed=4, scale=2) if sink else None
    if sink:
        s[0] = -math.inf               # as if there were none
    got = run_attention("cuda", torch.bfloat16, q, k, v, scale=d ** -0.5, size=size,
                        sink=s, parts=parts)
    # results are averages of values: one rounding of them and of the weights
    close(got, L.sink_attention(q, k, v, d ** -0.5, size, s), torch.bfloat16)


@pytest.mark.parametrize("H,G,d", [(32, 32, 64), (64, 32, 128)])
@pytest.mark.parametrize("parts", [(512,), (513,), (400, 120)], ids=str)
def test_as_many_blocks_as_units_and_more(H, G, d, parts):
    """8 and 9 tiles of 32 blocks, for which a page's keys are split or not."""
    T, size = sum(parts), 200
    q, k, v = rnd(T, H, d, seed=1), rnd(T, G, d, seed=2), rnd(T, G, d, seed=3)
    s = rnd(H, seed=4, scale=2)
    got = run_attention("cuda", torch.bfloat16, q, k, v, scale=d ** -0.5, size=size,
                        sink=s, parts=parts)
    i, j = torch.arange(T).unsqueeze(1), torch.arange(T)
    seen = (j <= i) & (j >= i - i % size)
    kk, vv = (t.repeat_interleave(H // G, 1).transpose(0, 1).double() for t in (k, v))
    x = q.transpose(0, 1).double() @ kk.transpose(1, 2) * d ** -0.5
    x = torch.cat([x.masked_fill(~seen, -math.inf), s.double().view(H, 1, 1).expand(H, T, 1)], 2)
    want = (torch.softmax(x, 2)[..., :-1] @ vv).transpose(0, 1)
    close(got, want.to(got.dtype).reshape(got.shape), torch.bfloat16)


@pytest.mark.parametrize("parts", [(65,), (64, 1)], ids=str)
def test_a_sink_that_is_no_number_shows(parts):
    """In its head, and in no other."""
    T, H, G, d = sum(parts), 4, 2, 64
    q, k, v = rnd(T, H, d, seed=1), rnd(T, G, d, seed=2), rnd(T, G, d, seed=3)
    sink = rnd(H, seed=4)
    sink[1] = math.nan
    got = run_attention("cuda", torch.bfloat16, q, k, v, scale=d ** -0.5, size=0,
                        sink=sink, parts=parts)
    assert got[:, 1].isnan().all()
    got[:, 1] = 0
    assert got.isfinite().all()


@pytest.mark.parametrize("H,G,d,e", [(4, 2, 64, 64), (3, 3, 128, 64),
                                     (64, 64, 64, 64), (128, 64, 128, 128)])
def test_a_sink_above_all_leaves_nothing(H, G, d, e):
    """Of its head, whether a page's keys are split (below 257 blocks) or not."""
    T = 290
    q, k, v = rnd(T, H, d, seed=1), rnd(T, G, d, seed=2), rnd(T, G, e, seed=3)
    sink = rnd(H, seed=4)
    sink[1] = math.inf
    got = run_attention("cuda", torch.bfloat16, q, k, v, scale=d ** -0.5, size=0,
                        sink=sink, parts=(T,))
    assert not got[:, 1].any()
    assert got.isfinite().all() and got[:, 0].any() and got[:, 2].any()
