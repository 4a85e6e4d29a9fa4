"""decode_attention against float64: rotation, cache append, attention of one
new token per row, at the edges of spans, tiles and depths."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(qkv, k, v, pos, tables, H):
    """Outputs and caches in float64; new keys are rounded as a cache holds
    them."""
    B, G, _, D = k.shape
    x = qkv.double().view(B, H + 2 * G, D)
    q, nk, nv = x[:, :H], x[:, H:H + G], x[:, H + G:]
    if tables is not None:
        c, s = (t.double()[pos].unsqueeze(1) for t in tables)

        def turn(t):
            u, w = t[..., 0::2], t[..., 1::2]
            return torch.stack([u * c - w * s, u * s + w * c], -1).flatten(2)

        q, nk = (turn(t).to(torch.bfloat16).double() for t in (q, nk))
    k, v = k.double().clone(), v.double().clone()
    out = torch.zeros(B, H, D, dtype=torch.float64, device=k.device)
    for b, p in enumerate(pos.tolist()):
        k[b, :, p], v[b, :, p] = nk[b], nv[b]
        kk, vv = (t[b, :, :p + 1].repeat_interleave(H // G, 0) for t in (k, v))
        w = torch.softmax((kk @ q[b].unsqueeze(2)).squeeze(2) / math.sqrt(D), 1)
        out[b] = (w.unsqueeze(1) @ vv).squeeze(1)
    return out.flatten(1), k, v


@pytest.mark.parametrize("D,H,G", [(128, 32, 8), (64, 12, 12), (64, 6, 3),
                                   (32, 4, 2), (128, 6, 2), (128, 8, 1)])
@pytest.mark.parametrize("L,depths", [
    (1, [0]), (64, [0, 63, 17]), (65, [64, 63, 1]), (1000, [999, 64, 128, 0]),
    (4096, [4095, 4094, 2047, 511, 512, 15, 16])])
@pytest.mark.parametrize("turn", [None, torch.float32, torch.bfloat16])
def test_matches_float64(D, H, G, L, depths, turn):
    from scaffold import ops

    torch.manual_seed(L + D)
    B, dev = len(depths), "cuda"
    qkv = torch.randn(B, (H + 2 * G) * D, device=dev).bfloat16()
    k, v = (torch.randn(B, G, L, D, device=dev).bfloat16() for _ in range(2))
    pos = torch.tensor(depths, device=dev)
    tables = None
    if turn is not None:
        tables = [t.to(turn) for t in ops.rope_tables(L, D, 1e4, dev)]
    want, wk, wv = _reference(qkv, k, v, pos, tables, H)
    for b, p in enumerate(depths):       # places not written yet
        k[b, :, p:] = float("nan")
        v[b, :, p:] = float("nan")
    got = ops.require_ext().decode_attention(
        qkv, k, v, pos, None, *(tables or (None, None)), H)
    # one rounding of the result, and of a turned query to its neighbour
    # where float32 and float64 fall on different sides: 2^-9 each
    err = (got.double() - want).norm() / want.norm()
    assert err < 2 * 2 ** -9, err
    for b, p in enumerate(depths):
        torch.testing.assert_close(k[b, :, p].double(), wk[b, :, p],
                                   rtol=2 ** -7, atol=1e-6)
        assert torch.equal(v[b, :, p].double(), wv[b, :, p])


def test_rows_left_alone_and_one_position_for_all():
    from scaffold import ops

    f = ops.require_ext().decode_attention
    torch.manual_seed(0)
    B, H, G, L, D = 5, 8, 2, 300, 64
    qkv = torch.randn(B, (H + 2 * G) * D, device="cuda").bfloat16()
    k, v = (torch.randn(B, G, L, D, device="cuda").bfloat16() for _ in range(2))
    k0, v0 = k.clone(), v.clone()
    active = torch.tensor([1, 0, 1, 1, 1], device="cuda")
    pos = torch.tensor([7, 8, L, -1, 299], device="cuda")
    got = f(qkv, k, v, pos, active, None, None, H)
    want = _reference(qkv[::4], k0[::4], v0[::4], pos[::4], None, H)[0]
    assert (got[::4].double() - want).norm() / want.norm() < 2 ** -8
    assert got[1].eq(0).all()                       # idle: nothing
    assert got[2].isnan().all() and got[3].isnan().all()  # no such place
    for t, t0 in ((k, k0), (v, v0)):
        assert torch.equal(t[1:4], t0[1:4])
    one = f(qkv, k0.clone(), v0.clone(), torch.tensor([41], device="cuda"),
            None, None, None, H)
    all_ = f(qkv, k0.clone(), v0.clone(), torch.full((B,), 41, device="cuda"),
             None, None, None, H)
    assert torch.equal(one, all_)


def test_far_scores_do_not_overflow():
    """A key that dwarfs all others in one span, and scores near the largest
    float's exponent range."""
    from scaffold import ops

    B, H, G, L, D = 1, 4, 1, 2048, 128
    torch.manual_seed(1)
    qkv = torch.randn(B, (H + 2 * G) * D, device="cuda").bfloat16() * 30
    k, v = (torch.randn(B, G, L, D, device="cuda").bfloat16() for _ in range(2))
    k[0, 0, 700] = qkv[0, :D] * 30
    pos = torch.tensor([L - 1], device="cuda")
    want = _reference(qkv, k, v, pos, None, H)[0]
    got = ops.require_ext().decode_attention(qkv, k, v, pos, None, None, None, H)
    assert (got.double() - want).norm() / want.norm() < 2 ** -8


def _inputs(L, H=4, G=2, D=128):
    torch.manual_seed(L)
    qkv = torch.randn(1, (H + 2 * G) * D, device="cuda").bfloat16()
    k, v = (torch.randn(1, G, L, D, device="cuda").bfloat16() for _ in range(2))
    return qkv, k, v


def _attend(qkv, k, v, depth, H=4):
    from scaffold import ops

    out = ops.require_ext().decode_attention(
        qkv, k, v, torch.tensor([depth], device="cuda"), None, None, None, H)
    return out.view(H, -1)


@pytest.mark.parametrize("L", [40, 4096])
@pytest.mark.parametrize("at", [0, 5, 30, "new"])
def test_a_score_that_is_no_number_shows(L, at):
    """NaN in one cached key, or in the new one, is NaN in the heads that see
    it, and in no other."""
    qkv, k, v = _inputs(L)
    if at == "new":
        qkv[0, 5 * 128 + 3] = float("nan")
    else:
        k[0, 1, at, 3] = float("nan")
    out = _attend(qkv, k, v, L - 2)
    assert out[:2].isfinite().all() and out[2:].isnan().all()


@pytest.mark.parametrize("L", [40, 4096])
@pytest.mark.parametrize("best", [3, 37, "new"])
def test_scores_far_below_zero(L, best):
    """Every score near the lowest float's exponent: the highest still wins."""
    qkv, k, v = _inputs(L)
    qkv[:, :512] = 1e17
    k[:] = -1e18
    qkv[:, 512:768] = -1e18
    if best == "new":
        qkv[:, 512:768] = -9e17
        want = qkv[0, 768:].view(2, 1, 128)
    else:
        k[:, :, best] = -9e17
        want = v[0, :, best].unsqueeze(1)
    out = _attend(qkv, k, v, L - 2)
    assert torch.equal(out.view(2, 2, 128), want.expand(2, 2, 128))
    k[:] = -1e30                         # -inf throughout: no weights at all
    qkv[:, :512] = 1e30
    qkv[:, 512:768] = -1e30
    assert _attend(qkv, k, v, L - 2).isnan().all()


@pytest.mark.parametrize("L", [18, 40, 49, 4096])
@pytest.mark.parametrize("back", [0, 1, 2, 17])
def test_infinite_values(L, back):
    """An infinite value, cached `back` places before the new one or new, is
    infinite in its column of the heads that see it, and nothing else is."""
    qkv, k, v = _inputs(L)
    if back == 0:
        qkv[0, 7 * 128 + 3] = float("inf")
    else:
        v[0, 1, L - 1 - back, 3] = float("inf")
    out = _attend(qkv, k, v, L - 1)
    assert (out[2:, 3] == float("inf")).all()
    out[2:, 3] = 0
    assert out.isfinite().all()


@pytest.mark.parametrize("D,H,G", [(128, 16, 2), (64, 18, 2), (32, 22, 1)])
@pytest.mark.parametrize("L", [33, 130, 1500])
def test_heads_that_share_keys(D, H, G, L):
    """More heads to a kv head than a block takes, fewer in its last, and
    depths around a tile of 32 keys and the tiles of a block of waves."""
    from scaffold import ops

    torch.manual_seed(L)
    depths = [d for d in (0, 30, 31, 32, 127, 128, 129, L - 1) if d < L]
    B = len(depths)
    qkv = torch.randn(B, (H + 2 * G) * D, device="cuda").bfloat16()
    k, v = (torch.randn(B, G, L, D, device="cuda").bfloat16() for _ in range(2))
    pos = torch.tensor(depths, device="cuda")
    want = _reference(qkv, k, v, pos, None, H)[0]
    for b, p in enumerate(depths):
        k[b, :, p:] = float("nan")
        v[b, :, p:] = float("nan")
    got = ops.require_ext().decode_attention(qkv, k, v, pos, None, None, None, H)
    # float32 sums and weights; one rounding of the result is at most 2^-9 of
    # each value
    assert (got.double() - want).norm() / want.norm() < 2 ** -9


@pytest.mark.parametrize("D,H,G", [(64, 1, 1), (64, 2, 1), (64, 3, 1), (128, 8, 2),
                                   (32, 8, 1)])
def test_weights_keep_the_bits_of_float32(D, H, G):
    """Two keys whose scores differ by a last bit, below a third one's: what is
    left of their values, 1 and -1, is the difference of two weights."""
    from scaffold import ops

    torch.manual_seed(0)
    R = 256
    q = torch.rand(R, device="cuda") / 4 + 0.25
    near = (torch.rand(R, device="cuda") + 1).bfloat16()
    best = (near + 8 + 24 * torch.rand(R, device="cuda")).bfloat16()
    qkv = torch.zeros(R, H + 2 * G, D, device="cuda").bfloat16()
    k, v = (torch.zeros(R, G, 3, D, device="cuda").bfloat16() for _ in range(2))
    qkv[:, :H, 0] = q[:, None].bfloat16()
    qkv[:, H:H + G, 0] = (near * (1 + 2 ** -7))[:, None]
    qkv[:, H + G:] = 1
    k[:, :, 0, 0] = best[:, None]
    k[:, :, 1, 0] = near[:, None]
    v[:, :, 1] = -1
    pos = torch.full((R,), 2, device="cuda")
    want = _reference(qkv.view(R, -1), k, v, pos, None, H)[0]
    got = ops.require_ext().decode_attention(qkv.view(R, -1), k, v, pos, None, None,
                                             None, H)
    # one rounding of the result is at most 2^-9 of it; 16 bits of the weights
    # alone would leave twice that of their difference
    assert (got.double() - want).norm() / want.norm() < 2 ** -9


@pytest.mark.parametrize("D,B,G,L", [
    (32, 3, 2, 256), (32, 3, 2, 257), (32, 64, 4, 1024), (32, 64, 4, 1100),
    (64, 3, 2, 256), (64, 3, 2, 257), (64, 51, 5, 300), (64, 64, 4, 300),
    (128, 3, 2, 256), (128, 64, 4, 256), (128, 64, 4, 511), (128, 64, 4, 512),
    (128, 2, 2, 2100)])
def test_two_heads_to_a_kv_head(D, B, G, L):
    """Sizes on both sides of where the matrix kernel takes over, and of where
    one span does."""
    from scaffold import ops

    torch.manual_seed(L)
    H = 2 * G
    qkv = torch.randn(B, (H + 2 * G) * D, device="cuda").bfloat16()
    k, v = (torch.randn(B, G, L, D, device="cuda").bfloat16() for _ in range(2))
    pos = torch.randint(0, L, (B,), device="cuda")
    pos[0], pos[-1] = L - 1, 0
    want, wk, wv = _reference(qkv, k, v, pos, None, H)
    for b, p in enumerate(pos.tolist()):
        k[b, :, p:] = float("nan")
        v[b, :, p:] = float("nan")
    got = ops.require_ext().decode_attention(qkv, k, v, pos, None, None, None, H)
    # float32 sums and weights; one rounding of the result is at most 2^-9 of
    # each value
    assert (got.double() - want).norm() / want.norm() < 2 ** -9
    for b, p in enumerate(pos.tolist()):
        assert torch.equal(k[b, :, p].double(), wk[b, :, p])
        assert torch.equal(v[b, :, p].double(), wv[b, :, p])


@pytest.mark.parametrize("H", [2, 4, 8])
def test_a_cache_without_places_is_refused(H):
    from scaffold import ops

    qkv = torch.zeros(1, (H + 4) * 64, device="cuda").bfloat16()
    k, v = (torch.zeros(1, 2, 0, 64, device="cuda").bfloat16() for _ in range(2))
    with pytest.raises(RuntimeError, match="places"):
        ops.require_ext().decode_attention(
            qkv, k, v, torch.zeros(1, dtype=torch.int64, device="cuda"), None, None, None, H)


@pytest.mark.parametrize("D,B,G,L", [
    (128, 33, 8, 4096), (128, 43, 6, 4100), (128, 44, 8, 4161), (128, 89, 4, 4096),
    (64, 257, 1, 8192)])
def test_a_few_more_blocks_than_compute_units(D, B, G, L):
    """Rows that fill the chip once and a little walk their keys in three spans;
    depths at the spans' edges, and rows whose later spans are empty."""
    from scaffold import ops

    torch.manual_seed(B + L)
    H, dev = 4 * G, "cuda"
    span = ((L + 63) // 64 + 2) // 3 * 64
    edges = [L - 1, 0, 1, span - 1, span, span + 1, 2 * span - 1, 2 * span, 63, 64]
    qkv = torch.randn(B, (H + 2 * G) * D, device=dev).bfloat16()
    k, v = (torch.randn(B, G, L, D, device=dev).bfloat16() for _ in range(2))
    pos = torch.randint(0, L, (B,), device=dev)
    pos[:len(edges)] = torch.tensor(edges, device=dev)
    got = ops.require_ext().decode_attention(qkv, k, v, pos, None, None, None, H)
    for r in range(0, B, 11):                 # float64 of a few rows at a time
        rows = slice(r, min(B, r + 11))
        want = _reference(qkv[rows], k[rows], v[rows], pos[rows], None, H)[0]
        # one rounding of the result: 2^-9
        err = (got[rows].double() - want).norm(dim=1) / want.norm(dim=1)
        assert err.max() < 2 * 2 ** -9, err
