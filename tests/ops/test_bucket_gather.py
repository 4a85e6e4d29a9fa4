"""Gradients that autograd made elsewhere come into their buckets: the copy
itself, and BucketedDDP on the GPU beside plain accumulation."""

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gather_into(dtype):
    from scaffold import ops

    torch.manual_seed(0)
    sizes = [1, 2, 7, 8, 9, 4096, 16384, 16385, 100003] + [3] * 70 + [0, 5]
    made = [torch.randn(n, device="cuda").to(dtype) for n in sizes]
    flat = torch.full((sum(sizes) + 1,), 9.0, device="cuda", dtype=dtype)
    places, at = [], 1                       # odd starts: nothing is aligned
    for n in sizes:
        places.append(flat[at:at + n])
        at += n
    # laid out differently on both sides, and the same but not contiguous
    made += [torch.randn(6, 5, device="cuda").to(dtype).t(),
             torch.randn(2, 3, 4, 5, device="cuda").to(dtype).contiguous(
                 memory_format=torch.channels_last)]
    places += [torch.zeros(5, 6, device="cuda", dtype=dtype),
               torch.zeros_like(made[-1])]
    ops.require_ext().gather_into(made, places)
    for m, p in zip(made, places):
        assert torch.equal(m, p)
    assert flat[0] == 9
    with pytest.raises(RuntimeError):
        ops.require_ext().gather_into([made[3]], [places[4]])


@pytest.mark.parametrize("n", [4, 100003])
def test_gather_into_goes_by_the_tensors_device(n):
    """Whichever device is current; without a GPU at hand, by torch's copies."""
    from scaffold import ops

    gather = ops.require_ext().gather_into
    gather([], [])
    last = torch.device("cuda", torch.cuda.device_count() - 1)
    for dev in (last, torch.device("cpu")):
        made = [torch.randn(n, device=dev), torch.randn(n).half()]
        places = [torch.zeros(n, device=dev), torch.zeros(n, device=dev)]
        with torch.cuda.device(0):
            gather(made, places)
        for m, p in zip(made, places):
            assert torch.equal(m.to(dev).float(), p)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_gradients_of_another_stream_live_until_they_are_read(dtype):
    """What was made on a side stream is dropped at once, and that stream gets
    memory of the same size while the copy still waits."""
    from scaffold import ops

    side = torch.cuda.Stream()
    n = 1 << 20
    places = [torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda")]
    with torch.cuda.stream(side):
        made = [torch.full((n,), 3.0, device="cuda", dtype=dtype) for _ in places]
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda._sleep(50_000_000)
    ops.require_ext().gather_into(made, places)
    del made
    with torch.cuda.stream(side):
        others = [torch.full((n,), 5.0, device="cuda", dtype=dtype)
                  for _ in range(4)]
    torch.cuda.synchronize()
    assert all(p.eq(3).all() for p in places) and others[0].eq(5).all()


class _Net(nn.Module):
    def __init__(self):
        super().__init__()
        self.emb = nn.Embedding(11, 24)
        self.conv = nn.Conv2d(1, 6, 3, padding=1, bias=False)
        self.a = nn.Linear(24, 24)
        self.b = nn.Linear(24, 11, bias=False)
        self.b.weight = self.emb.weight          # used twice
        self.unused = nn.Parameter(torch.randn(7))

    def forward(self, t):
        x = self.emb(t)
        x = x + self.conv(x.unsqueeze(1)).mean(1)
        return self.b(torch.tanh(self.a(x))).square().mean()


def _nets():
    from scaffold.dist.ddp import BucketedDDP

    torch.manual_seed(1)
    net = _Net().cuda().to(memory_format=torch.channels_last)
    ref = _Net().cuda().to(memory_format=torch.channels_last)
    ref.load_state_dict(net.state_dict())
    return BucketedDDP(net, bucket_cap_mb=0.002, first_bucket_mb=0.0005), ref


def _check(ddp, ref):
    for b in ddp.buckets:
        for p, v in zip(b.params, b.views):
            assert p.grad is v                   # views, whoever made them
    for (n, p), q in zip(ddp.module.named_parameters(), ref.parameters()):
        want = torch.zeros_like(q) if q.grad is None else q.grad
        torch.testing.assert_close(p.grad, want, rtol=1e-5, atol=1e-7, msg=n)


def test_steps_and_accumulation():
    ddp, ref = _nets()
    t = [torch.randint(0, 11, (4, 24), device="cuda") for _ in range(3)]
    for step in range(3):
        ddp.zero_grad()
        ref.zero_grad()
        with ddp.no_sync():
            ddp(t[0]).backward()
        ref(t[0]).backward()
        _check(ddp, ref)                         # also between micro-steps
        if step:
            with ddp.no_sync():
                ddp(t[1]).backward()
            ref(t[1]).backward()
        ddp(t[2]).backward()
        ddp.finish()
        ref(t[2]).backward()
        _check(ddp, ref)
    # without zero_grad a step adds to what is there
    ddp(t[0]).backward()
    ddp.finish()
    ref(t[0]).backward()
    _check(ddp, ref)
    # and without a backward there are zeros
    ddp.zero_grad()
    ddp.finish()
    assert all(b.flat.eq(0).all() for b in ddp.buckets)


def test_overlap_off_and_grads_dropped_by_the_user():
    ddp, ref = _nets()
    ddp.overlap = False
    t = torch.randint(0, 11, (4, 24), device="cuda")
    for p in ddp.module.parameters():
        p.grad = None
    ddp(t).backward()
    ddp.finish()
    ref(t).backward()
    _check(ddp, ref)


def test_captured_step():
    """A step in a graph fills the same buckets on every replay."""
    ddp, ref = _nets()
    t = torch.randint(0, 11, (4, 24), device="cuda")

    def step():
        ddp.zero_grad()
        ddp(t).backward()
        ddp.finish()

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    for i in range(3):
        t.copy_(torch.randint(0, 11, t.shape, device="cuda"))
        for b in ddp.buckets:
            b.flat.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        ref.zero_grad()
        ref(t).backward()
        _check(ddp, ref)


class _TwoStreams(nn.Module):
    """Two layers of one bucket, one of them on a side stream that is late."""

    def __init__(self):
        super().__init__()
        self.a, self.b = (nn.Linear(256, 256, bias=False) for _ in range(2))
        self.side = None

    def forward(self, x):
        if self.side is None:
            return (self.a(x) * self.b(x)).sum()
        cur = torch.cuda.current_stream()
        self.side.wait_stream(cur)
        with torch.cuda.stream(self.side):
            u = _Late.apply(self.a(x))
        v = self.b(x)
        cur.wait_stream(self.side)
        return (u * v).sum()


class _Late(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, dy):
        torch.cuda._sleep(20_000_000)
        return dy * 1


@pytest.mark.parametrize("overlap", [True, False])
def test_gradients_of_several_streams(overlap):
    from scaffold.dist.ddp import BucketedDDP

    torch.manual_seed(5)
    net = _TwoStreams().cuda()
    ref = _TwoStreams().cuda()
    ref.load_state_dict(net.state_dict())
    net.side = torch.cuda.Stream()
    ddp = BucketedDDP(net, overlap=overlap)
    for _ in range(3):
        x = torch.randn(64, 256, device="cuda")
        ddp.zero_grad()
        ddp(x).backward()
        ddp.finish()
        got = [p.grad.clone() for p in net.parameters()]
        ref.zero_grad()
        ref(x).backward()
        for g, p in zip(got, ref.parameters()):
            torch.testing.assert_close(g, p.grad)


def test_one_stream_launches_from_the_backward():
    """The overlap is still there where a bucket has one stream."""
    ddp, _ = _nets()
    t = torch.randint(0, 11, (4, 24), device="cuda")
    seen = []
    launch = ddp._launch
    ddp._launch = lambda b: seen.append(b.index) or launch(b)
    side = torch.cuda.Stream()
    for s in (torch.cuda.current_stream(), side):
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            ddp.zero_grad()
            del seen[:]
            ddp(t).backward()
            early = len(seen)
            ddp.finish()
        assert early >= len(ddp.buckets) - 1 > 0     # one param is unused
    torch.cuda.synchronize()
