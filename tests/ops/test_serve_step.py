"""The serving step of GPT-2 and Llama that one call issues, and the prompt
attention in it, at the edges of tiles and rules."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H,G", [(128, 8, 2), (64, 3, 3), (64, 8, 2)])
@pytest.mark.parametrize("S,Sk", [(1, 1), (2, 130), (63, 63), (64, 65),
                                  (256, 256), (257, 300), (700, 1025),
                                  # keys in two groups of waves, one with a tile more
                                  (1, 321), (130, 449), (257, 640), (500, 500)])
def test_prompt_attention_matches_float64(D, H, G, S, Sk):
    """Queries by token, keys and values in a cache with more behind them, heads that
    share keys."""
    from scaffold import ops

    torch.manual_seed(S + D)
    B, L = 2, Sk + 3
    q = torch.randn(B, S, H, D, device="cuda").bfloat16().transpose(1, 2)
    k, v = (torch.randn(B, G, L, D, device="cuda").bfloat16() for _ in range(2))
    v += 1                       # a mean: errors of the weights do not cancel
    k[:, :, Sk:] = float("nan")
    v[:, :, Sk:] = float("nan")
    got = ops.require_ext().prompt_attention(q, k, v, Sk).double()
    kk, vv = (t[:, :, :Sk].double().repeat_interleave(H // G, 1)
              for t in (k, v))
    s = q.double() @ kk.transpose(2, 3).contiguous() / math.sqrt(D)
    see = (torch.arange(Sk, device="cuda")
           <= torch.arange(Sk - S, Sk, device="cuda").unsqueeze(1))
    want = torch.softmax(s.masked_fill(~see, -math.inf), -1) @ vv
    # the result's rounding alone: half of 2^-8 at worst, 0.29 of it on
    # average; the weights' 16 bits and float32 sums are far below
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13).all()
    assert (got - want).norm() / want.norm() < 2.0 ** -9


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,S,Sk", [
    (1, 2, 2, 320), (1, 2, 2, 321),       # five tiles of keys, and a sixth
    (2, 3, 130, 385), (1, 2, 449, 449),   # one group has a tile more
    (1, 1, 1025, 1025),
    (8, 8, 512, 512), (8, 8, 513, 513)])  # 256 and 320 blocks
def test_prompt_keys_in_two_groups(D, B, H, S, Sk):
    from scaffold import ops

    torch.manual_seed(S + D)
    f = ops.require_ext().prompt_attention
    q, k, v = (torch.randn(B, H, n, D, device="cuda").bfloat16() for n in (S, Sk, Sk))
    v += 1
    got = f(q, k, v, Sk).double()
    s = q.double() @ k.double().transpose(2, 3).contiguous() / math.sqrt(D)
    see = (torch.arange(Sk, device="cuda")
           <= torch.arange(Sk - S, Sk, device="cuda").unsqueeze(1))
    want = torch.softmax(s.masked_fill(~see, -math.inf), -1) @ v.double()
    # the bounds of test_prompt_attention_matches_float64
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13).all()
    assert (got - want).norm() / want.norm() < 2.0 ** -9
    # all scores near the lowest float's exponent, the highest in either group's tiles
    q, k = torch.full_like(q, 1e17), torch.full_like(k, -1e18)
    for best in (0, 64, 70, 130):
        if best > Sk - S:
            break
        k[:, :, best] = -9e17
        got = f(q, k, v, Sk)
        assert torch.equal(got, v[:, :, best:best + 1].expand_as(got))
        k[:, :, best] = float("nan")
        assert f(q, k, v, Sk).isnan().all()
        k[:, :, best] = -1e18
    assert f(q * 1e13, k * 1e13, v, Sk).isnan().all()


@pytest.mark.parametrize("D,H,G", [(128, 4, 2), (64, 3, 3)])
@pytest.mark.parametrize("S,Sk", [(1, 70), (5, 5), (64, 65), (257, 300)])
def test_prompt_scores_far_below_zero(D, H, G, S, Sk):
    """Every score near the lowest float's exponent, the highest two keys back
    (or the first): what follows a row is not seen, and -inf is NaN."""
    from scaffold import ops

    f = ops.require_ext().prompt_attention
    torch.manual_seed(S)
    q = torch.full((2, H, S, D), 1e17, device="cuda").bfloat16()
    k = torch.full((2, G, Sk, D), -1e18, device="cuda").bfloat16()
    v = torch.randn(2, G, Sk, D, device="cuda").bfloat16()
    best = max(Sk - S - 2, 0)
    k[:, :, best] = -9e17
    want = v[:, :, best].repeat_interleave(H // G, 1).unsqueeze(2)
    got = f(q, k, v, Sk)
    assert torch.equal(got, want.expand_as(got))
    assert f(q * 1e13, k * 1e13, v, Sk).isnan().all()
    k[0, 0, best] = float("nan")
    got = f(q, k, v, Sk)
    assert got[0, :H // G].isnan().all() and got[0, H // G:].isfinite().all()
    assert got[1].isfinite().all()


def _model(name, **kw):
    from scaffold.config import load_config
    from scaffold.models import build_model

    keys = {"name": name, "vocab_size": 1003, "n_layers": 3, "n_heads": 4,
            "d_model": 256, "max_seq_len": 200, **kw}
    torch.manual_seed(3)
    m = build_model(load_config(None, [f"model.{k}={v}"
                                       for k, v in keys.items()]))
    with torch.no_grad():
        for n, p in m.named_parameters():
            if p.dim() == 1:
                p.add_(torch.randn_like(p) * 0.1)
            else:
                p.mul_(2)
    return m.bfloat16().eval()


@pytest.mark.parametrize("name,kw", [
    ("gpt2", {}), ("gpt2", {"d_ff": 520}),
    ("llama", {"n_kv_heads": 2, "d_ff": 520}),
    ("llama", {"n_kv_heads": 1, "d_ff": 8200}),
    ("llama", {"n_heads": 8, "n_kv_heads": 1, "d_ff": 520}),
    ("llama", {"n_heads": 10, "n_kv_heads": 2, "d_model": 640, "d_ff": 520})])
@pytest.mark.parametrize("B", [1, 7, 17, 65])
def test_step_matches_float32(name, kw, B):
    """A step at unequal depths and one at a common depth, against the
    block-by-block step of the same weights in float32 on the CPU."""
    from scaffold.generate import Generator

    m = _model(name, **kw)
    ref = Generator(_model(name, **kw).float())
    gen = Generator(m.cuda())
    L = 150
    cpu, gpu = ref.new_cache(B, L), gen.new_cache(B, L)
    for i in range(3):
        for a, b in ((cpu.k[i], gpu.k[i]), (cpu.v[i], gpu.v[i])):
            b.copy_(torch.randn_like(b, dtype=torch.float32))
            a.copy_(b)
    tok = torch.randint(0, 1003, (B, 1))
    pos = torch.randint(0, L, (B,))
    with torch.no_grad():
        assert gen._native_step(tok.cuda(), gpu, pos.cuda()) is not None
        got = gen.decode_step_varpos(tok.cuda(), gpu, pos.cuda()).cpu().float()
        want = ref.decode_step_varpos(tok, cpu, pos)
        # a bf16 stream: about ten roundings of 2^-9 a layer, independent
        assert (got - want).norm() / want.norm() < 3 * 2 ** -7
        cpu.len = gpu.len = 20
        got = gen._forward_tokens(tok.cuda(), gpu, 20).cpu().float()
        want = ref._forward_tokens(tok, cpu, 20)
        assert (got - want).norm() / want.norm() < 3 * 2 ** -7
        assert gpu.len == cpu.len == 21


# residual products of 16 MB of weights, whose depth is split over blocks and whose
# parts the next norm adds up
WIDE = [("llama", {"n_heads": 8, "n_kv_heads": 2, "d_model": 1024, "d_ff": 8200}),
        ("gpt2", {"n_heads": 8, "d_model": 1024, "d_ff": 8200})]


@pytest.mark.parametrize("name,kw", WIDE)
@pytest.mark.parametrize("B", [9, 17, 64])
def test_split_products_of_a_step(name, kw, B):
    from scaffold.generate import Generator

    kw = {**kw, "n_layers": 2, "vocab_size": 64}
    ref = Generator(_model(name, **kw).float())
    gen = Generator(_model(name, **kw).cuda())
    cpu, gpu = ref.new_cache(B, 40), gen.new_cache(B, 40)
    for a, b in zip(cpu.k + cpu.v, gpu.k + gpu.v):
        b.copy_(torch.randn_like(b, dtype=torch.float32))
        a.copy_(b)
    tok, pos = torch.randint(0, 64, (B, 1)), torch.randint(0, 40, (B,))
    with torch.no_grad():
        want = ref.decode_step_varpos(tok, cpu, pos)
        got = gen._native_step(tok.cuda(), gpu, pos.cuda()).cpu().float()
    # a bf16 stream: about ten roundings of 2^-9 a layer, independent
    assert (got - want).norm() / want.norm() < 3 * 2 ** -7


@pytest.mark.parametrize("name,kw", WIDE)
@pytest.mark.parametrize("B,S", [(1, 9), (3, 20), (2, 32), (12, 3)])
@pytest.mark.parametrize("every", [False, True])
def test_split_products_of_a_prompt(name, kw, B, S, every):
    """Without all logits the last layer's rows are fewer than the others',
    and as few as take whole depths."""
    from scaffold.generate import Generator

    kw = {**kw, "n_layers": 2, "vocab_size": 64}
    ref = Generator(_model(name, **kw).float())
    gen = Generator(_model(name, **kw).cuda())
    cpu, gpu = ref.new_cache(B, 40), gen.new_cache(B, 40)
    ids = torch.randint(0, 64, (B, S))
    with torch.no_grad():
        want = ref._forward_tokens(ids, cpu, 0, all_logits=every)
        got = gen._native_step(ids.cuda(), gpu, None, 0, all_logits=every)
    # a bf16 stream: about ten roundings of 2^-9 a layer, independent
    assert (got.cpu().float() - want).norm() / want.norm() < 3 * 2 ** -7


@pytest.mark.parametrize("rows,width,ff,splits", [
    (8, 1024, 8200, 0), (9, 1024, 8200, 2), (64, 1024, 8200, 2), (65, 1024, 8200, 0),
    (16, 7168, 2048, 4), (17, 7168, 2048, 0), (16, 8192, 2048, 0)])
def test_which_products_are_split(rows, width, ff, splits):
    """The rule itself, by the kernels that a step of two layers launches."""
    from torch.profiler import ProfilerActivity, profile

    from scaffold.generate import Generator

    gen = Generator(_model("llama", n_heads=width // 128, n_kv_heads=2, n_layers=2,
                           vocab_size=64, d_model=width, d_ff=ff).cuda())
    cache = gen.new_cache(rows, 8)
    tok = torch.zeros(rows, 1, dtype=torch.int64, device="cuda")
    pos = torch.zeros(rows, dtype=torch.int64, device="cuda")
    with torch.no_grad(), profile(activities=[ProfilerActivity.CUDA],
                                  acc_events=True) as prof:
        assert gen._native_step(tok, cache, pos) is not None
        torch.cuda.synchronize()
    names = [e.name for e in prof.events()]
    assert any("row_norm_kernel" in n for n in names)
    assert sum("skinny_split_kernel" in n for n in names) == splits


def test_step_is_left_to_the_blocks():
    """Routed feed-forwards and float32 models keep the general step."""
    from scaffold.generate import Generator

    tok = torch.zeros(2, 1, dtype=torch.int64, device="cuda")
    pos = torch.tensor([3, 4], device="cuda")
    for m in (_model("gpt2", n_experts=2), _model("gpt2").float()):
        gen = Generator(m.cuda())
        cache = gen.new_cache(2, 16)
        assert gen._native_step(tok, cache, pos) is None
        assert gen.decode_step_varpos(tok, cache, pos).isfinite().all()


def test_unknown_token_shows():
    from scaffold.generate import Generator

    gen = Generator(_model("gpt2").cuda())
    cache = gen.new_cache(2, 16)
    out = gen.decode_step_varpos(torch.tensor([[5], [1003]], device="cuda"),
                                 cache, torch.tensor([0, 0], device="cuda"))
    assert out[0].isfinite().all() and out[1].isnan().all()


@pytest.mark.parametrize("name,kw", [
    ("gpt2", {"n_heads": 4}), ("llama", {"n_kv_heads": 2, "d_ff": 520}),
    ("llama", {"n_heads": 2, "n_kv_heads": 1, "d_ff": 520}),
    ("llama", {"n_heads": 10, "n_kv_heads": 2, "d_model": 640, "d_ff": 520})])
@pytest.mark.parametrize("B,S,p0", [(1, 2, 0), (3, 5, 0), (2, 9, 64),
                                    (1, 130, 20), (2, 64, 1), (1, 1, 0)])
@pytest.mark.parametrize("every", [False, True])
def test_prompt_matches_float32(name, kw, B, S, p0, every):
    """A prompt, or what follows one, against float32 on the CPU: logits and
    the keys and values it leaves."""
    from scaffold.generate import Generator

    m = _model(name, **kw)
    ref = Generator(_model(name, **kw).float())
    gen = Generator(m.cuda())
    L = 150
    cpu, gpu = ref.new_cache(B, L), gen.new_cache(B, L)
    for i in range(3):
        for a, b in ((cpu.k[i], gpu.k[i]), (cpu.v[i], gpu.v[i])):
            b.copy_(torch.randn_like(b, dtype=torch.float32))
            a.copy_(b)
    cpu.len = gpu.len = p0
    tok = torch.randint(0, 1003, (B, S))
    with torch.no_grad():
        assert gen._native_step(tok.cuda(), gpu, None, p0) is not None
        want = ref._forward_tokens(tok, cpu, p0, all_logits=every)
        got = gen._forward_tokens(tok.cuda(), gpu, p0, all_logits=every)
    assert got.shape == want.shape and gpu.len == cpu.len == p0 + S
    # a bf16 stream: about ten roundings of 2^-9 a layer, independent
    assert (got.cpu().float() - want).norm() / want.norm() < 3 * 2 ** -7
    for a, b in zip(cpu.k + cpu.v, gpu.k + gpu.v):
        b = b.cpu().float()
        new = slice(p0, p0 + S)
        err = (a[:, :, new] - b[:, :, new]).norm() / a[:, :, new].norm()
        assert err < 3 * 2 ** -7
        assert torch.equal(a[:, :, :p0], b[:, :, :p0])
        assert torch.equal(a[:, :, p0 + S:], b[:, :, p0 + S:])


def test_prompt_that_does_not_fit_is_refused():
    from scaffold.generate import Generator

    gen = Generator(_model("llama", n_kv_heads=2, d_ff=520).cuda())
    cache = gen.new_cache(1, 8)
    with torch.no_grad(), pytest.raises(RuntimeError):
        gen._forward_tokens(torch.zeros(1, 9, dtype=torch.int64,
                                        device="cuda"), cache, 0)


@pytest.mark.parametrize("name,kw", [("gpt2", {}),
                                     ("llama", {"n_kv_heads": 2, "d_ff": 520})])
def test_parametrized_weights_are_left_to_the_blocks(name, kw):
    """Unmerged adapters, whose merged weights would all be alive in one call:
    layer by layer, and the step of the merged model."""
    from scaffold.generate import Generator
    from scaffold.lora import LoRAAdapter, apply_lora, merge_lora

    m = _model(name, **kw).cuda()
    apply_lora(m, r=4)
    for mod in m.modules():
        if isinstance(mod, LoRAAdapter):
            torch.nn.init.normal_(mod.B, std=0.02)
    gen = Generator(m)
    tok = torch.tensor([[5], [9]], device="cuda")
    pos = torch.tensor([0, 3], device="cuda")
    with torch.no_grad():
        assert gen._native_step(tok, gen.new_cache(2, 16), pos) is None
        got = gen.decode_step_varpos(tok, gen.new_cache(2, 16), pos)
        cache = gen.new_cache(2, 16)
        ids = torch.arange(10, device="cuda").view(2, 5)
        prompt = gen._forward_tokens(ids, cache, 0)
    gen = Generator(merge_lora(m).eval())
    with torch.no_grad():
        assert gen._native_step(tok, gen.new_cache(2, 16), pos) is not None
        want = gen.decode_step_varpos(tok, gen.new_cache(2, 16), pos)
        merged = gen._forward_tokens(ids, gen.new_cache(2, 16), 0)
    # two bf16 streams of the same weights: see test_step_matches_float32
    for g, w in ((got, want), (prompt, merged)):
        assert (g.float() - w.float()).norm() / w.float().norm() < 6 * 2 ** -7


@pytest.mark.parametrize("name,kw,embeddings", [
    ("gpt2", {}, ("wte", "wpe")),
    ("llama", {"n_kv_heads": 2, "d_ff": 520}, ("embed",))])
def test_embeddings_that_do_more_than_look_up(name, kw, embeddings):
    """Hooks fire, an own forward is called, and their results count."""
    from scaffold.generate import Generator

    tok = torch.tensor([[5], [9]], device="cuda")
    ids = torch.arange(6, device="cuda").view(2, 3)
    pos = torch.tensor([3, 3], device="cuda")

    @torch.no_grad()
    def run(m):
        gen, out = Generator(m), []
        cache = gen.new_cache(2, 16)
        out.append(gen._forward_tokens(ids, cache, 0))
        out.append(gen.decode_step_varpos(tok, cache, pos))
        return out, gen._native_step(tok, cache, pos)

    for attr in embeddings:
        m = _model(name, **kw).cuda()
        mod, table = getattr(m, attr), getattr(m, attr).weight.detach().clone()
        plain, native = run(m)
        assert native is not None
        hits = []
        ways = []
        h = mod.register_forward_hook(lambda *a: hits.append(1))
        ways.append(run(m))
        assert len(hits) == 2
        h.remove()
        h = mod.register_forward_pre_hook(lambda *a: hits.append(1))
        ways.append(run(m))
        assert len(hits) == 4
        h.remove()
        h = torch.nn.modules.module.register_module_forward_hook(
            lambda a, *b: hits.append(1) if a is mod else None)
        ways.append(run(m))
        assert len(hits) == 6
        h.remove()
        mod.forward = lambda t: torch.nn.functional.embedding(t, table)
        ways.append(run(m))
        del mod.forward
        for out, native in ways:
            assert native is None
            for g, w in zip(out, plain):
                assert (g.float() - w.float()).norm() / w.float().norm() < 6 * 2 ** -7
        h = mod.register_forward_hook(lambda m, a, out: out * 0 + 1)
        ones = run(m)[0]
        h.remove()
        assert not any(torch.equal(g, w) for g, w in zip(ones, ways[0][0]))
        assert run(m)[1] is not None


@pytest.mark.parametrize("name,kw", [
    ("gpt2", {}), ("llama", {"n_kv_heads": 2, "d_ff": 512}),
    ("llama", {"n_heads": 16, "n_kv_heads": 2, "d_model": 512, "d_ff": 512})])
@pytest.mark.parametrize("rank", [0, 1])
def test_a_shard_steps_as_on_the_cpu(name, kw, rank):
    """One rank's share of a tensor-parallel model (partial sums, since no
    group is there to add them): layer by layer, attention in one launch."""
    from scaffold.dist.tp import shard_llama_tp
    from scaffold.generate import Generator

    ref = Generator(shard_llama_tp(_model(name, **kw), rank, 2).float())
    gen = Generator(shard_llama_tp(_model(name, **kw), rank, 2).cuda())
    cpu, gpu = ref.new_cache(3, 40), gen.new_cache(3, 40)
    ids = torch.randint(0, 1003, (3, 9))
    tok, pos = torch.randint(0, 1003, (3, 1)), torch.tensor([9, 4, 9])
    with torch.no_grad():
        assert gen._native_step(tok.cuda(), gpu, pos.cuda()) is None
        want = [ref._forward_tokens(ids, cpu, 0),
                ref.decode_step_varpos(tok, cpu, pos)]
        got = [gen._forward_tokens(ids.cuda(), gpu, 0),
               gen.decode_step_varpos(tok.cuda(), gpu, pos.cuda())]
    for g, w in zip(got, want):
        # a bf16 stream: about ten roundings of 2^-9 a layer, independent
        assert (g.cpu().float() - w).norm() / w.norm() < 3 * 2 ** -7
    for a, b in zip(cpu.k + cpu.v, gpu.k + gpu.v):
        assert (a - b.cpu().float()).norm() / a.norm() < 3 * 2 ** -7


@pytest.mark.parametrize("name,kw", [
    ("gpt2", {"n_heads": 4}), ("llama", {"n_heads": 4, "n_kv_heads": 2,
                                         "d_model": 512, "d_ff": 520})])
@pytest.mark.parametrize("B,S,Sk", [
    (1, 2, 4999), (1, 2, 5000), (2, 9, 5003),   # by the number of keys
    (1, 660, 5000), (1, 670, 5000),             # by rows: heads of 64
    (1, 700, 5000), (1, 710, 5000)])            # heads of 128
def test_few_rows_before_many_keys(name, kw, B, S, Sk):
    """Portions on both sides of the rule that takes the float32 products,
    against float32 on the CPU."""
    from scaffold.generate import Generator

    kw = {**kw, "max_seq_len": 5100, "n_layers": 2, "vocab_size": 64}
    ref = Generator(_model(name, **kw).float())
    gen = Generator(_model(name, **kw).cuda())
    cpu, gpu = ref.new_cache(B, Sk + 1), gen.new_cache(B, Sk + 1)
    for a, b in zip(cpu.k + cpu.v, gpu.k + gpu.v):
        b.copy_(torch.randn_like(b, dtype=torch.float32))
        a.copy_(b)
        b[:, :, Sk:] = float("nan")
    p0 = cpu.len = gpu.len = Sk - S
    ids = torch.randint(0, 64, (B, S))
    with torch.no_grad():
        want = ref._forward_tokens(ids, cpu, p0, all_logits=True)
        assert gen._native_step(ids.cuda(), gpu, None, p0) is not None
        got = gen._forward_tokens(ids.cuda(), gpu, p0, all_logits=True)
    # a bf16 stream: about ten roundings of 2^-9 a layer, independent
    assert (got.cpu().float() - want).norm() / want.norm() < 3 * 2 ** -7


@pytest.mark.parametrize("name,kw,S,Sk,products", [
    ("gpt2", {}, 2, 4999, False), ("gpt2", {}, 2, 5000, True),
    ("gpt2", {}, 667, 5000, True), ("gpt2", {}, 668, 5000, False),
    ("llama", {"n_kv_heads": 2, "d_model": 512, "d_ff": 520}, 704, 5000, True),
    ("llama", {"n_kv_heads": 2, "d_model": 512, "d_ff": 520}, 705, 5000, False)])
def test_which_rows_take_the_float32_products(name, kw, S, Sk, products):
    """The rule itself, by the library calls that a step makes."""
    from scaffold.generate import Generator

    gen = Generator(_model(name, **kw, max_seq_len=5100, n_layers=2,
                           vocab_size=64).cuda())
    cache = gen.new_cache(1, Sk + 1)
    for t in cache.k + cache.v:
        t.zero_()
    ids = torch.zeros(1, S, dtype=torch.int64, device="cuda")
    with torch.no_grad(), torch.autograd.profiler.profile() as prof:
        assert gen._native_step(ids, cache, None, Sk - S, all_logits=True) is not None
    calls = [e.key for e in prof.key_averages()]
    assert ("aten::softmax" in calls) == products


@pytest.mark.parametrize("name", ["gpt2", "llama"])
def test_products_of_a_prompt_are_seen_by_modes(name):
    """Under a mode that watches calls, products of many rows stay torch's."""
    from torch.utils._python_dispatch import TorchDispatchMode

    from scaffold.generate import Generator

    class Watch(TorchDispatchMode):
        products = 0

        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            self.products += f.overloadpacket.__name__ in ("mm", "addmm", "linear")
            return f(*args, **(kwargs or {}))

    gen = Generator(_model(name, d_ff=1024).cuda())
    ids = torch.zeros(1, 128, dtype=torch.int64, device="cuda")
    with torch.no_grad(), Watch() as watch:
        assert gen._native_step(ids, gen.new_cache(1, 128), None, 0, all_logits=True) is not None
    assert watch.products == 3 * 4 + 1       # of a layer, and the head's
