"""The head of a vocabulary that is no multiple of eight: logits and gradients
in rows of whole lines."""

import pytest
import torch
import torch.nn.functional as F

from scaffold import ops

pytestmark = pytest.mark.gpu


def _made(R, V, K):
    torch.manual_seed(R)
    x = torch.randn(R, K, device="cuda").bfloat16().requires_grad_()
    w = (torch.randn(V, K, device="cuda") / K ** 0.5).bfloat16().requires_grad_()
    return x, w, torch.randint(0, V, (R,), device="cuda")


def _gradient(x, w, t):
    """The gradient of the logits, whose bits no layout changes."""
    m = ops.require_ext()
    logits = m.head_logits(x.detach(), w.detach())
    return m.softmax_xent_bwd(logits, t, m.softmax_xent_fwd(logits, t)[1])


def _close(got, a, b):
    """got = a b, of which every partial sum is below the sum of sizes: the
    result's rounding, and that of depth / 32 + 32 float32 sums."""
    a, b = a.double().contiguous(), b.double()
    want, size = a @ b, a.abs() @ b.abs()
    lim = 2.0 ** -8 * want.abs() + (a.shape[1] / 32 + 32) * 2.0 ** -24 * size
    assert got.shape == want.shape and ((got.double() - want).abs() <= lim).all()


def _calls(monkeypatch):
    ext, calls = ops.require_ext(), []
    made = ext.head_grads
    monkeypatch.setattr(ext, "head_grads", lambda *a: calls.append(1) or made(*a))
    return calls


SIZES = [(2047, 10001, 256),      # both gradients by the library
         (16384, 3001, 768),      # dx by the kernel
         (2048, 15001, 768),      # dW by the kernel
         (2049, 15007, 768)]


@pytest.mark.parametrize("R,V,K", SIZES)
def test_each_number_of_each_step(R, V, K):
    """The last rows and columns too, which are not whole eights: every logit, weight and
    gradient against 64 bits, of the operands that its step was given."""
    m = ops.require_ext()
    x, w, t = _made(R, V, K)
    x, w = x.detach(), w.detach()
    logits = m.head_logits(x, w)
    assert logits.shape == (R, V) and logits.stride() == (-(-V // 128) * 128, 1)
    _close(logits, x, w.t())
    loss, lse = m.softmax_xent_fwd(logits, t)
    z = logits.double()
    want = z.logsumexp(1)
    # sums of V exponentials that are 2^-21 off, by 256 threads; logarithms below 2^5
    off = (V / 256 + 40) * 2.0 ** -24
    assert ((lse.double() - want).abs() <= off).all()
    at = z.gather(1, t.unsqueeze(1)).squeeze(1)
    assert ((loss.double() - (want - at)).abs() <= 2 * off).all()
    d = m.softmax_xent_bwd(logits, t, lse)
    assert d.stride() == logits.stride()
    p = (z - want.unsqueeze(1)).exp()
    want = p.scatter_add(1, t.unsqueeze(1), torch.full((R, 1), -1.0, device="cuda").double())
    assert ((d.double() * R - want).abs() <= 2.0 ** -8 * want.abs() + 2 * off * p).all()
    # which their gradients' products read
    assert not d.as_strided((R, d.stride(0) - V), d.stride(), V).any()
    dx, dw = m.head_grads(d, x, w, True, True)
    _close(dx, d, w)
    _close(dw, d.t(), x)


@pytest.mark.parametrize("R,V,K", SIZES)
def test_loss_and_gradients(R, V, K, monkeypatch):
    calls = _calls(monkeypatch)
    x, w, t = _made(R, V, K)
    loss = ops.lm_head_ce(x.view(1, R, K), w, t)
    got = torch.autograd.grad(loss, (x, w), torch.tensor(3.0, device="cuda"))
    assert calls
    u, v = (s.detach().double().requires_grad_() for s in (x, w))
    want_loss = F.cross_entropy(u @ v.t(), t)
    want = torch.autograd.grad(3 * want_loss, (u, v))
    assert abs(loss.item() - want_loss.item()) < 1e-3
    for g, h in zip(got, want):
        assert g.shape == h.shape and g.is_contiguous()
        # logits rounded to 8 bits move each weight by 2^-9 |logit|, gradients once more
        assert (g.double() - h).norm() < 0.01 * h.norm()
    # what lies between the rows does not count, frozen operands cost nothing
    (only,) = torch.autograd.grad(ops.lm_head_ce(x, w.detach(), t), x)
    assert (3 * only.double() - want[0]).norm() < 0.01 * want[0].norm()
    with torch.no_grad():
        assert abs(ops.lm_head_ce(x, w, t).item() - loss.item()) < 1e-6


def test_as_near_as_one_row_behind_the_other(monkeypatch):
    """Sums in another order: one rounding of 2^-9 in some hundred values."""
    calls = _calls(monkeypatch)
    x, w, t = _made(16384, 3001, 768)
    a = torch.autograd.grad(ops.lm_head_ce(x, w, t), (x, w))
    assert calls
    b = torch.autograd.grad(ops.softmax_cross_entropy(F.linear(x, w), t), (x, w))
    for g, h in zip(a, b):
        assert (g.double() - h.double()).norm() < 1e-3 * h.double().norm()


@pytest.mark.parametrize("R,V,K", [(2047, 10001, 256), (2048, 15001, 768)])
@pytest.mark.parametrize("how", ["host", "copy", "strides"])
def test_saved_tensors_that_hooks_have_copied(R, V, K, how):
    """Logits come back with one row behind the other, or as they were: the
    gradients are the products they were."""
    from torch.autograd.graph import save_on_cpu, saved_tensors_hooks

    x, w, t = _made(R, V, K)
    with {"host": save_on_cpu(),
          "copy": saved_tensors_hooks(lambda s: s.clone(memory_format=torch.contiguous_format),
                                      lambda s: s),
          "strides": saved_tensors_hooks(
              lambda s: s.clone(memory_format=torch.contiguous_format),
              lambda s: F.pad(s, (0, 24))[..., :-24] if s.shape == (R, V) else s)}[how]:
        loss = ops.lm_head_ce(x, w, t)
    dx, dw = torch.autograd.grad(loss, (x, w))
    d = _gradient(x, w, t)
    _close(dx, d, w.detach())
    _close(dw, d.t(), x.detach())


def test_small_or_other_operands_go_the_general_way(monkeypatch):
    calls = _calls(monkeypatch)
    ext = ops.require_ext()
    made = ext.head_logits
    monkeypatch.setattr(ext, "head_logits", lambda x, w: (
        calls.append(1) if w.shape[0] % 8 == 0 or len(x) < 1000 else None, made(x, w))[1])
    for R, V, K, dtype in ((100, 3001, 768, torch.bfloat16), (16384, 3000, 768, torch.bfloat16),
                           (16384, 301, 768, torch.float32)):
        x, w, t = _made(R, V, K)
        x, w = (s.detach().to(dtype).requires_grad_() for s in (x, w))
        torch.autograd.grad(ops.lm_head_ce(x, w, t), (x, w))
    assert not calls


def test_a_graph_of_the_gradients(monkeypatch):
    calls = _calls(monkeypatch)
    x, w, t = _made(2047, 10001, 256)
    (dx,) = torch.autograd.grad(ops.lm_head_ce(x, w, t), x, create_graph=True)
    assert not calls and torch.autograd.grad(dx.float().sum(), w)[0].any()
