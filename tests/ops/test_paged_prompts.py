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


def _check(H, G, d, e, parts, size=0, sink=None, slopes=None):
    T = sum(parts)
    q, k, v = rnd(T, H, d, seed=1), rnd(T, G, d, seed=2), rnd(T, G, e, seed=3)
    got = run_attention("cuda", torch.bfloat16, q, k, v, scale=d ** -0.5, size=size,
                        sink=sink, parts=parts, slopes=slopes).double()
    i, j = torch.arange(T, device="cuda").unsqueeze(1), torch.arange(T, device="cuda")
    q, k, v = (t.transpose(0, 1).cuda() for t in (
        q, k.repeat_interleave(H // G, 1), v.repeat_interleave(H // G, 1)))
    x = q @ k.transpose(1, 2).contiguous() * d ** -0.5
    if slopes is not None:
        x = x - slopes.cuda().double().view(H, 1, 1) * (i - j)
    x = x.masked_fill((j > i) | (j < i - i % size if size else j < 0), -math.inf)
    none = torch.full((H,), -math.inf).double()
    s = (none if sink is None else sink).cuda().view(H, 1, 1).expand(H, T, 1)
    w = torch.softmax(torch.cat([x, s], 2), 2)[..., :-1]
    want = (w @ v).transpose(0, 1)
    # one rounding of the result; weights in two parts of 8 bits, the bias and the
    # exponents of scores below 2^7 in float32
    lim = 2.0 ** -8 * want.abs() + 2.0 ** -14 * (w @ v.abs()).transpose(0, 1) + 2.0 ** -20
    assert ((got - want).abs() <= lim).all()


FORMS = [(16, 4, 128, 128), (4, 2, 64, 64), (8, 2, 64, 128), (4, 2, 128, 64), (6, 3, 72, 104),
         (3, 3, 128, 128), (3, 1, 64, 64), (5, 5, 64, 128), (3, 3, 128, 64), (3, 3, 104, 40)]


@pytest.mark.parametrize("H,G,d,e", FORMS)
@pytest.mark.parametrize("parts", [(64,), (65,), (256,), (257,), (30, 34, 33, 40)], ids=str)
def test_few_pages(H, G, d, e, parts):
    """As many pages as are not split yet, and one more: one (and none, values of 64), or
    four with two heads a block."""
    _check(H, G, d, e, parts, sink=rnd(H, seed=4, scale=2))
    _check(H, G, d, e, parts, size=70, slopes=torch.rand(H) / 8)


@pytest.mark.parametrize("H,G,d,e", FORMS)
@pytest.mark.parametrize("what", ["plain", "sink", "none", "chunks", "slopes"])
def test_many_blocks(H, G, d, e, what):
    """More blocks than compute units, where pages are not split: as many copies of the
    form's groups of heads as it takes for 5 and 9 tiles."""
    for parts in ((257,), (60, 515)):
        n = 257 // -(-max(parts) // 64) // G + 1
        sink = rnd(n * H, seed=4, scale=2) if what in ("sink", "none", "chunks") else None
        if what == "none":
            sink[::2] = -math.inf
        _check(n * H, n * G, d, e, parts, size=200 if what == "chunks" else 0, sink=sink,
               slopes=torch.rand(n * H) / 8 if what == "slopes" else None)


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
