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
