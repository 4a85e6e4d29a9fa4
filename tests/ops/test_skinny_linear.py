"""Products of few rows with a weight matrix, at the edges of tiles, spans and
rules."""

import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(1, 8), (15, 24), (16, 128), (50, 768),
                                 (768, 3072), (6150, 136), (20483, 64),
                                 (4096, 1032)])
@pytest.mark.parametrize("M", [1, 8, 16, 17, 33, 64])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_matches_float64(N, K, M, act):
    from scaffold import ops

    torch.manual_seed(N + K + M)
    dev = "cuda"
    x = torch.randn(M, K + 8, device=dev).bfloat16()[:, :K]
    w = (torch.randn(N * (2 if act == 2 else 1), K, device=dev)
         / math.sqrt(K)).bfloat16()
    b = None if act == 2 else torch.randn(N, device=dev).bfloat16()
    r = torch.randn(M, N, device=dev).bfloat16()
    got = ops.require_ext().skinny_linear(x, w, b, r, act).double()
    y = x.double() @ w.double().T
    if act == 2:
        y = F.silu(y[:, :N]) * y[:, N:]
    else:
        y = y + b.double()
    if act == 1:
        y = F.gelu(y, approximate="tanh")
    y = y + r.double()
    # one rounding of the result (2^-9 of it); sums of K products and the
    # exponential in float32 are far below
    assert ((got - y).abs() <= 2.0 ** -8 * y.abs() + 2.0 ** -14).all()


@pytest.mark.parametrize("M,N,K", [
    (2, 1028, 776), (3, 1024, 136), (4, 1025, 2056), (4, 2048, 264),
    (2, 2052, 1000), (2, 6144, 2064), (2, 6148, 2064), (1, 7001, 2048),
    (5, 2048, 72), (7, 2049, 200), (8, 4100, 2080)])
@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("off", [0, 2])
def test_places_of_the_depth(M, N, K, act, off):
    """Up to 8 rows: the edges of what takes four or two places of the depth at
    once, depths that do not fill them, bias and residual in and out of line."""
    from scaffold import ops

    torch.manual_seed(N + K + M)
    dev = "cuda"
    x = torch.randn(M, K + 8, device=dev).bfloat16()[:, :K]
    w = (torch.randn(N * (2 if act == 2 else 1), K, device=dev)
         / math.sqrt(K)).bfloat16()
    b = None if act == 2 else torch.randn(N + off, device=dev).bfloat16()[off:]
    r = torch.randn(M, N + off, device=dev).bfloat16()[:, off:]
    got = ops.require_ext().skinny_linear(x, w, b, r, act).double()
    y = x.double() @ w.double().T
    if act == 2:
        y = F.silu(y[:, :N]) * y[:, N:]
    else:
        y = y + b.double()
    if act == 1:
        y = F.gelu(y, approximate="tanh")
    y = y + r.double()
    # as above
    assert ((got - y).abs() <= 2.0 ** -8 * y.abs() + 2.0 ** -14).all()


@pytest.mark.parametrize("M,K", [(1, 8), (1, 4096), (2, 4096), (3, 768),
                                 (10, 768), (16, 504), (16, 512), (9, 520),
                                 (4, 4096), (5, 1024), (8, 2040), (16, 1024)])
@pytest.mark.parametrize("N,act", [(48, 0), (2304, 1), (6150, 2), (20483, 0)])
@pytest.mark.parametrize("kind", ["layer", "rms"])
def test_norm_of_the_rows(M, K, N, act, kind):
    from scaffold import ops

    torch.manual_seed(N + K + M)
    dev = "cuda"
    x = (torch.randn(M, K + 8, device=dev) * 3 + 1).bfloat16()[:, :K]
    w = (torch.randn(N * (2 if act == 2 else 1), K, device=dev)
         / math.sqrt(K)).bfloat16()
    nw = torch.randn(K, device=dev).bfloat16()
    nb = torch.randn(K, device=dev).bfloat16() if kind == "layer" else None
    got = ops.require_ext().skinny_linear(
        x, w, None, None, act, norm_w=nw, norm_b=nb, eps=1e-5).double()
    xd = x.double()
    if nb is not None:
        h = F.layer_norm(xd, (K,), nw.double(), nb.double(), 1e-5)
    else:
        h = F.rms_norm(xd, (K,), nw.double(), 1e-5)
    y = h @ w.double().T
    # rounding of the normed rows: 2^-9 of each term, 8 deviations of their sum
    d = 2.0 ** -9 * 8 * ((h * h) @ (w.double() ** 2).T).sqrt() / math.sqrt(3)
    if act == 2:
        g, u = y[:, :N], y[:, N:]
        y = F.silu(g) * u
        d = 1.1 * d[:, :N] * (u.abs() + d[:, N:]) + F.silu(g).abs() * d[:, N:]
    elif act == 1:
        y, d = F.gelu(y, approximate="tanh"), 1.13 * d
    assert ((got - y).abs() <= d + 2.0 ** -8 * y.abs() + 2.0 ** -14).all()


def test_refuses_what_it_is_not_for():
    from scaffold import ops

    f = ops.require_ext().skinny_linear
    x = torch.zeros(65, 64, device="cuda", dtype=torch.bfloat16)
    w = torch.zeros(16, 64, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        f(x, w)                            # too many rows
    with pytest.raises(RuntimeError):
        f(x[:4, :12], w[:, :12].contiguous())   # depth not in eights
    with pytest.raises(RuntimeError):
        f(x[:4].float(), w.float())
    with pytest.raises(RuntimeError):
        f(x[:4, 4:12], w[:, :8].contiguous())   # rows not aligned
    with pytest.raises(RuntimeError):       # more than the kernel norms
        f(torch.zeros(17, 64, device="cuda", dtype=torch.bfloat16), w,
          norm_w=w[0])
    with pytest.raises(RuntimeError):
        f(x[:4], w, norm_w=w[0, :8])


@pytest.mark.parametrize("N,K", [(4096, 2056), (1028, 8200), (20484, 416),
                                 (2048, 14336)])
@pytest.mark.parametrize("M", [9, 16, 17, 32, 33, 64])
def test_parts_of_the_depth(N, K, M):
    """Spans and chunks that do not divide the depth, rows of w that do not
    fill a block; what lies behind the depth is not read into the sums."""
    from scaffold import ops

    torch.manual_seed(N + K + M)
    dev = "cuda"
    x = torch.randn(M, K + 8, device=dev).bfloat16()[:, :K]
    x.as_strided((M, 8), (K + 8, 1), K).fill_(float("nan"))
    w = torch.randn(N, K, device=dev).bfloat16()
    b = torch.randn(N, device=dev).bfloat16()
    got = ops.require_ext().skinny_linear_parts(x, w, b)
    assert got.shape[0] > 1 or K < 512 or N > 8192
    y = x.double() @ w.double().T + b.double()
    # K / 32 sums after each other and one over 32, each rounded to 2^-24 of
    # at most the sum of the terms' sizes
    d = (K / 32 + 32 + 8) * 2.0 ** -24 * (x.abs().double() @ w.abs().double().T
                                         + b.abs().double())
    assert ((got.double().sum(0) - y).abs() <= d).all()


def test_an_infinite_weight_stays_infinite():
    from scaffold import ops

    x = torch.ones(9, 4104, device="cuda", dtype=torch.bfloat16)
    w = torch.ones(2048, 4104, device="cuda", dtype=torch.bfloat16)
    w[3, -1] = float("inf")
    got = ops.require_ext().skinny_linear_parts(x, w).sum(0)
    assert (got[:, 3] == float("inf")).all()
    got[:, 3] = 0
    assert got.isfinite().all()
