"""One token a row over pages, against float64: infinite values, float32
weights, more heads to a kv head than a block takes, deep caches."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

PAGE = 64


def rnd(*shape):
    return torch.randn(*shape, device="cuda").bfloat16()


class Rows:
    """Rows at depths `pos` over caches of their own, of which nothing behind
    the cached keys is a number; `shared`: the pages before the last are."""

    def __init__(self, H, G, d, e, pos, shared=False):
        self.H, self.G, self.d, self.e, self.pos = H, G, d, e, pos
        n = max(pos) // PAGE + 1
        R = len(pos)
        own = torch.arange(R * n).view(R, n)
        if shared:
            for r, p in enumerate(pos):
                own[r, :p // PAGE] = torch.arange(p // PAGE)
                own[r, p // PAGE] = n + r
        used = int(own.max()) + 1 if shared else R * n
        self.table = own.int().cuda()
        self.k, self.v = rnd(used, G, PAGE, d), rnd(used, G, PAGE, e)
        for r, p in enumerate(pos):
            self.k[own[r, p // PAGE], :, p % PAGE:] = float("nan")
            self.v[own[r, p // PAGE], :, p % PAGE:] = float("nan")
        self.qkv = rnd(R, (H + G) * d + G * e)

    def parts(self, r):
        """q (H, d), keys (G, p + 1, d), values of row r, the new one last."""
        q, k, v = self.qkv[r].split([self.H * self.d, self.G * self.d, self.G * self.e])
        p, pages = self.pos[r], self.table[r, :self.pos[r] // PAGE + 1].long()
        cached = [c[pages].transpose(0, 1).flatten(1, 2)[:, :p] for c in (self.k, self.v)]
        return (q.view(self.H, self.d), torch.cat([cached[0], k.view(self.G, 1, -1)], 1),
                torch.cat([cached[1], v.view(self.G, 1, -1)], 1))

    def run(self, scale, size=0, qw=None, kw=None, slopes=None, eps=1e-6):
        from scaffold.ops.lm import require_lm_ext

        R = len(self.pos)
        none = torch.empty(0, 4, dtype=torch.int32, device="cuda")
        out = require_lm_ext().paged_attention(
            self.qkv, self.k.clone(), self.v.clone(), self.table,
            torch.tensor(self.pos, device="cuda").int(),
            torch.arange(R, device="cuda").int(), none, R, qw, kw, None, slopes,
            self.H, size, scale, eps, max(self.pos) + 1)
        return out.view(R, self.H, self.e)


def weights(q, k, scale, slopes=None):
    """(H, keys) of q (H, d) and k (G, keys, d), the last of which is q's."""
    k = k.double().repeat_interleave(q.shape[0] // k.shape[0], 0)
    s = (k * q.double().unsqueeze(1)).sum(-1) * scale
    if slopes is not None:
        back = torch.arange(k.shape[1] - 1, -1, -1, device="cuda")
        s = s - slopes.double().unsqueeze(1) * back
    return torch.softmax(s, -1)


@pytest.mark.parametrize("H,G,d,e", [(4, 2, 128, 128), (6, 2, 64, 40), (8, 2, 32, 64)])
@pytest.mark.parametrize("L", [18, 40, 65, 129, 1000])
@pytest.mark.parametrize("back", [0, 1, 2, 17])
@pytest.mark.parametrize("value", [math.inf, -math.inf])
def test_infinite_values(H, G, d, e, L, back, value):
    """An infinite value, cached `back` places before the new one or new, is
    infinite in its column of the heads that see it, and nothing else is."""
    torch.manual_seed(L)
    x = Rows(H, G, d, e, [L - 1])
    if back == 0:
        x.qkv[0, (H + G) * d + e + 3] = value
    else:
        x.v[x.table[0, (L - 1 - back) // PAGE].long(), 1, (L - 1 - back) % PAGE, 3] = value
    out = x.run(d ** -0.5)[0]
    assert (out[H // G:, 3] == value).all()
    out[H // G:, 3] = 0
    assert out.isfinite().all()


@pytest.mark.parametrize("H,G,d,e", [(3, 1, 64, 64), (4, 2, 128, 128)])
def test_weights_keep_the_bits_of_float32(H, G, d, e):
    """Two keys whose scores differ by a last bit, below a third one's: what is
    left of their values, 1 and -1, is the difference of two weights."""
    torch.manual_seed(0)
    R = 256
    x = Rows(H, G, d, e, [2] * R)
    q, near = torch.rand(R, device="cuda") / 4 + 0.25, torch.rand(R, device="cuda") + 1
    near = near.bfloat16()
    best = (near + 8 + 24 * torch.rand(R, device="cuda")).bfloat16()
    for t in (x.qkv, x.k, x.v):
        t.zero_()
    cell = x.table[:, 0].long()
    x.k[cell, :, 0, 0] = best[:, None]
    x.k[cell, :, 1, 0] = near[:, None]
    x.v[cell, :, 1] = -1
    rows = x.qkv[:, :H * d].view(R, H, d)
    rows[:, :, 0] = q[:, None].bfloat16()
    x.qkv[:, H * d:(H + G) * d].view(R, G, d)[:, :, 0] = (near * (1 + 2 ** -7))[:, None]
    x.qkv[:, (H + G) * d:] = 1
    got = x.run(d ** -0.5)
    want = torch.empty(R, H, dtype=torch.double, device="cuda")
    for r in range(R):
        q_, k_, _ = x.parts(r)
        w = weights(q_, k_, d ** -0.5)
        want[r] = w[:, 2] - w[:, 1]
    # one rounding of the result is at most 2^-9 of it; 16 bits of the weights
    # alone would leave twice that of their difference
    assert (got.double() - want.unsqueeze(2)).norm() / (want.norm() * e ** 0.5) < 2 ** -9


@pytest.mark.parametrize("H,G,d,e", [(17, 1, 64, 64), (80, 2, 128, 72), (33, 1, 40, 128)])
@pytest.mark.parametrize("pos", [[0, 31, 32, 200], [700]])
def test_more_heads_than_a_block_takes(H, G, d, e, pos):
    """Norms and a bias by distance among them; the new key is appended once."""
    torch.manual_seed(H)
    x = Rows(H, G, d, e, pos)
    qw, kw = rnd(d) / 4 + 1, rnd(d) / 4 + 1
    slopes = torch.rand(H, device="cuda") / 8
    got = x.run(0.2, qw=qw, kw=kw, slopes=slopes, eps=0.01)

    def norm(t, w):
        t = t.double()
        return (t * (t.pow(2).mean(-1, keepdim=True) + 0.01).rsqrt() * w.double()).bfloat16()

    for r in range(len(pos)):
        q, k, v = x.parts(r)
        k = torch.cat([k[:, :-1], norm(k[:, -1:], kw)], 1)
        w = weights(norm(q, qw), k, 0.2, slopes)
        want = torch.einsum("hk,hke->he", w, v.double().repeat_interleave(H // G, 0))
        # one rounding of the result, at most 2^-9 of each value, and one of a
        # normed element that float32 and float64 round to either side, 2^-8 of
        # one of its d products
        assert (got[r].double() - want).norm() / want.norm() < 2 ** -8


def test_more_than_a_wave_knows_the_pages_of():
    """Depths behind 8192 keys in one split."""
    torch.manual_seed(5)
    H, G, d, e = 8, 4, 16, 8
    x = Rows(H, G, d, e, [8400 - 3 * r for r in range(64)], shared=True)
    got = x.run(1.0)
    for r in (0, 1, 31, 63):
        q, k, v = x.parts(r)
        want = torch.einsum("hk,hke->he", weights(q, k, 1.0),
                            v.double().repeat_interleave(H // G, 0))
        assert (got[r].double() - want).norm() / want.norm() < 2 ** -8
