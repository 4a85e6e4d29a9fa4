"""The last rows of a prompt behind a quarter of a million keys: what float32's
sums over so many weights lose."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

KEYS, ROWS, HEADS, DIM = 1 << 18, 8, 4, 128


def inputs():
    """q (HEADS, ROWS, DIM), k and v (HEADS, KEYS, DIM) and the exact result:
    the first key is a row's best, all others weigh the same, and every column
    of the values has two of them, 3 : 4."""
    torch.manual_seed(0)
    q, k = (torch.zeros(HEADS, n, DIM, device="cuda") for n in (ROWS, KEYS))
    q[..., 0] = torch.linspace(0.5, 8, ROWS, device="cuda")
    k[:, :, 0] = -1
    k[:, 0, 0] = 1
    a, b = (torch.rand(HEADS, 1, DIM, device="cuda") + 0.5 for _ in range(2))
    third = (torch.arange(KEYS, device="cuda") % 7 < 3).view(1, -1, 1)
    q, k, v = (t.bfloat16() for t in (q, k, torch.where(third, a, b)))
    w = torch.exp(-2 * q[0, :, 0].double() / math.sqrt(DIM))     # of a key but the first
    seen = torch.arange(KEYS - ROWS + 1, KEYS + 1, device="cuda")
    first = ((seen + 6) // 7 + (seen + 5) // 7 + (seen + 4) // 7).double()
    a, b = v[:, 0].double(), v[:, 3].double()
    w, first, seen = (t.view(1, -1, 1) for t in (w, first, seen.double()))
    num = a[:, None] * (1 + w * (first - 1)) + b[:, None] * w * (seen - first)
    return q, k, v, num / (1 + w * (seen - 1))


def check(got, want):
    # A row's factor, whose deviation the results' own roundings make 2^-13.
    # Values: 2^15 products of 16 keys and a part of their weights, one added
    # after the other, each rounded to 2^-24 of a running sum, all alike at worst:
    # 2^-10.  Weights added up by tiles come to 2^-12, one after the other, of
    # which a lane has 2^17, to 2^-8 at worst, and 2^-9 here.
    f = (got.double() * want).sum((0, 2)) / (want * want).sum((0, 2)) - 1
    assert f.abs().max() < 2.0 ** -10


def test_dense_cache():
    from scaffold import ops

    q, k, v, want = inputs()
    check(ops.require_ext().prompt_attention(q[None], k[None], v[None], KEYS)[0], want)


def test_pages():
    from scaffold.ops.lm import require_lm_ext

    q, k, v, want = inputs()
    kc, vc = (t.view(HEADS, -1, 64, DIM).transpose(0, 1).contiguous() for t in (k, v))
    new = slice(KEYS - ROWS, KEYS)
    qkv = torch.cat([t.transpose(0, 1).flatten(1) for t in (q, k[:, new], v[:, new])], 1)
    ints = dict(dtype=torch.int32, device="cuda")
    got = require_lm_ext().paged_attention(
        qkv.contiguous(), kc, vc, torch.arange(KEYS // 64, **ints).view(1, -1),
        torch.arange(new.start, new.stop, **ints), torch.zeros(ROWS, **ints),
        torch.tensor([[0, ROWS, new.start, 0]], **ints), 0, None, None, None, None,
        HEADS, 0, DIM ** -0.5, 1e-6, KEYS)
    check(got.view(ROWS, HEADS, DIM).transpose(0, 1), want)
