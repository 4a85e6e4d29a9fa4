"""BucketedDDP — the in-repo data-parallel engine (contract C4).

Design, MI355X-first:

* **Gradient-as-bucket-view**: each bucket owns ONE contiguous flat
  buffer; every param's ``.grad`` is a view into it once its bucket is
  reduced.  On the GPU ``zero_grad`` only lets go of the views: autograd
  then hands over the gradients as they are made, and one launch per
  bucket copies them in (two passes over memory per gradient; clearing
  the buffer and adding to it are four, in a launch per parameter).
  Gradients that accumulate (``no_sync``) go into the views in place.
* **Bucket partition in reverse parameter order** (grads become ready
  roughly in reverse-forward order during backward), with a small first
  bucket so the first all-reduce fires early.
* **Overlap**: when a bucket's last grad accumulates
  (``register_post_accumulate_grad_hook``), its SUM all-reduce is
  launched ``async_op=True``.  ProcessGroupNCCL (RCCL on ROCm) orders
  the collective against the compute stream and runs it on its own
  stream, so it proceeds concurrently with the remaining backward
  kernels over xGMI.  ``finish()`` waits all works (stream-ordered, no
  host sync).
* A bucket whose gradients are made on several streams waits for
  ``finish()``: there the caller's stream is behind all of them.
* **Averaging** is folded into the optimizer's fused AdamW
  ``grad_scale=1/world`` (one less full-gradient pass).
* Bucket sizes default to 25 MiB, first bucket 4 MiB — chosen so that
  >=7 RCCL channels (one per xGMI link) stay busy; sweepable via
  ``dist.bucket_cap_mb`` (bench harness mode).
"""

from __future__ import annotations

import contextlib
from dataclasses import dataclass, field
from typing import Dict, List, Optional

import torch
import torch.nn as nn

from .. import ops
from .comm import Comm


@dataclass
class GradBucket:
    index: int
    params: List[torch.nn.Parameter]
    flat: torch.Tensor = None  # type: ignore[assignment]
    views: List[torch.Tensor] = field(default_factory=list)
    pending: int = 0
    work: object = None
    launched: bool = False
    ready: bool = False
    stream: Optional[int] = None         # where its first gradient was made
    mixed: bool = False                  # others on another stream

    @property
    def numel(self) -> int:
        return sum(p.numel() for p in self.params)

    @property
    def nbytes(self) -> int:
        return self.flat.numel() * self.flat.element_size()


def partition_buckets(
    params: List[torch.nn.Parameter],
    bucket_cap_mb: float,
    first_bucket_mb: float,
) -> List[List[torch.nn.Parameter]]:
    """Split params (REVERSED construction order) into size-capped groups.

    Pure function — unit-tested on CPU (SURVEY §4 unit tier).
    """
    # Buckets must be dtype-homogeneous (one flat comm buffer per bucket).
    # Partition each dtype's params as its own stream (reverse order kept)
    # instead of splitting at every dtype flip — a bf16 model with fp32
    # BatchNorm params interleaved would otherwise shatter into ~2x-per-
    # layer tiny buckets.  Readiness hooks make cross-stream ordering safe.
    streams: Dict[torch.dtype, List[torch.nn.Parameter]] = {}
    for p in reversed(params):
        streams.setdefault(p.dtype, []).append(p)

    buckets: List[List[torch.nn.Parameter]] = []
    for plist in streams.values():
        cur: List[torch.nn.Parameter] = []
        cur_bytes = 0
        cap = first_bucket_mb * (1 << 20) if not buckets else bucket_cap_mb * (1 << 20)
        for p in plist:
            p_bytes = p.numel() * p.element_size()
            if cur and cur_bytes + p_bytes > cap:
                buckets.append(cur)
                cur = []
                cur_bytes = 0
                cap = bucket_cap_mb * (1 << 20)
            cur.append(p)
            cur_bytes += p_bytes
        if cur:
            buckets.append(cur)
    return buckets


def _gather_into(made, places) -> None:
    """What gather_into does on the GPU: gradients into the views of a bucket.
    One that lies in the bucket itself is left where it is the view under
    another name (p.grad = p.grad.detach()), else copied out before others are
    copied in."""
    own = places[0].untyped_storage().data_ptr()
    todo = []
    for g, v in zip(made, places):
        if g.layout != torch.strided:
            # torch's add of a sparse tensor to a view misses the view's place
            # in its storage
            g = g.to_dense()
        elif g.untyped_storage().data_ptr() == own:
            if g.data_ptr() == v.data_ptr() and g.stride() == v.stride():
                continue
            g = g.clone()
        todo.append((g, v))
    for g, v in todo:
        v.copy_(g)


class BucketedDDP(nn.Module):
    def __init__(
        self,
        module: nn.Module,
        comm: Optional[Comm] = None,
        bucket_cap_mb: float = 25,
        first_bucket_mb: float = 4,
        overlap: bool = True,
    ):
        super().__init__()
        self.module = module
        self.comm = comm if comm is not None else Comm()
        self.overlap = overlap
        self._sync_enabled = True
        self._require_finish = False

        # params marked _no_ddp are RANK-LOCAL by design (expert-parallel
        # MoE shards: each rank owns different experts) — they join
        # neither the buckets nor the wrap-time broadcast
        self.trainable = [p for p in module.parameters()
                          if p.requires_grad
                          and not getattr(p, "_no_ddp", False)]
        self.local_params = [p for p in module.parameters()
                             if p.requires_grad
                             and getattr(p, "_no_ddp", False)]

        # 1) rank-0 params/buffers win (SURVEY §3.1 broadcast at wrap)
        if self.comm.is_distributed:
            with torch.no_grad():
                for t in list(module.parameters()) + list(module.buffers()):
                    if getattr(t, "_no_ddp", False):
                        continue
                    if t.is_floating_point() or t.dtype in (torch.int64, torch.int32):
                        self.comm.broadcast(t.data, src=0)

        # 2) buckets + flat buffers + grad views
        groups = partition_buckets(self.trainable, bucket_cap_mb, first_bucket_mb)
        self.buckets: List[GradBucket] = []
        self._param_bucket: Dict[int, GradBucket] = {}
        for i, group in enumerate(groups):
            numel = sum(p.numel() for p in group)
            dtype = group[0].dtype
            device = group[0].device
            flat = torch.zeros(numel, dtype=dtype, device=device)
            b = GradBucket(index=i, params=group, flat=flat)
            off = 0
            for p in group:
                # as_strided matches the param's layout (channels_last conv
                # weights are dense permutations, not C-contiguous)
                view = flat[off : off + p.numel()].as_strided(p.shape, p.stride())
                p.grad = view  # autograd accumulates in place into the bucket
                b.views.append(view)
                self._param_bucket[id(p)] = b
                off += p.numel()
            b.pending = len(group)
            self.buckets.append(b)

        self._next_launch = 0  # index-ordered collective issue cursor

        # 3) readiness hooks
        self._hooks = [
            p.register_post_accumulate_grad_hook(self._make_hook(p))
            for p in self.trainable
        ]

    # ------------------------------------------------------------- hooks
    def _make_hook(self, p: torch.nn.Parameter):
        def hook(param: torch.Tensor) -> None:
            if not self._sync_enabled:
                return
            b = self._param_bucket[id(p)]
            b.pending -= 1
            if b.flat.is_cuda:
                # a copy out of this hook is in line with gradients of its own
                # stream alone; behind the backward the caller's stream is
                # with those of all
                s = torch._C._cuda_getCurrentRawStream(b.flat.device.index)
                if b.stream is None:
                    b.stream = s
                elif b.stream != s:
                    b.mixed = True
            if b.pending == 0 and self.overlap and not b.mixed:
                b.ready = True
                self._launch_ready_in_order()

        return hook

    def _launch_ready_in_order(self) -> None:
        """Launch ready buckets strictly by INDEX.  Collectives on one
        communicator must be issued in the same order on every rank or
        NCCL-class backends can mismatch/deadlock; autograd readiness
        order is not guaranteed identical across ranks, so a bucket
        that becomes ready early waits for its predecessors (same rule
        as torch DDP's reducer).  Buckets are partitioned in reverse
        parameter order, so index order ~= expected readiness order and
        the wait is normally empty."""
        while self._next_launch < len(self.buckets):
            b = self.buckets[self._next_launch]
            if not b.ready:
                return
            self._launch(b)
            self._next_launch += 1

    def _collect(self, b: GradBucket) -> None:
        """Bring gradients that autograd made elsewhere into the bucket:
        every .grad is its view afterwards."""
        made, places = [], []
        for p, v in zip(b.params, b.views):
            g = p.grad
            if g is v:
                continue
            if g is None:                # took no part in this backward
                v.zero_()
            else:
                made.append(g)
                places.append(v)
            p.grad = v
        if made:
            with torch.no_grad():
                if b.flat.is_cuda:
                    ops.require_ext().gather_into(made, places)
                else:
                    _gather_into(made, places)

    def _launch(self, b: GradBucket) -> None:
        if b.launched:
            return
        self._collect(b)
        if hasattr(self.comm, "all_reduce_bucket"):
            # direct-RCCL path: enqueued on the dedicated comm stream,
            # joined once in finish() (no per-bucket Work objects)
            self.comm.all_reduce_bucket(b.flat)
        else:
            b.work = self.comm.all_reduce(b.flat, async_op=True)
        b.launched = True

    # -------------------------------------------------------------- API
    def forward(self, *args, **kwargs):
        if self._sync_enabled:
            self._require_finish = True
        return self.module(*args, **kwargs)

    def finish(self) -> None:
        """End-of-backward: launch stragglers, wait all reduce works."""
        if not self._sync_enabled:
            return
        for b in self.buckets:
            if not b.launched:
                self._launch(b)
        if hasattr(self.comm, "join"):
            self.comm.join()  # compute stream waits comm stream, no host sync
        for b in self.buckets:
            if b.work is not None:
                b.work.wait()  # stream-ordered on RCCL; host wait on gloo
        self._reset()
        self._require_finish = False

    def _reset(self) -> None:
        for b in self.buckets:
            b.pending = len(b.params)
            b.work = None
            b.launched = False
            b.ready = False
            b.stream = None
            b.mixed = False
        self._next_launch = 0

    def zero_grad(self) -> None:
        """Start from no gradients.  On the GPU the params let go of their
        views and the buckets are filled anew (_collect): until then .grad
        is None and a bucket's flat buffer holds what it held.  On the CPU
        the flat buffers are zeroed.  Rank-local params (_no_ddp, e.g. EP
        experts) own ordinary .grad tensors — drop them too, or they
        silently ACCUMULATE across steps (found via a resume-divergence
        hunt: the accumulated history is exactly what a checkpoint cannot
        restore)."""
        for b in self.buckets:
            if not b.flat.is_cuda:
                b.flat.zero_()
                continue
            for p in b.params:
                p.grad = None
        for p in self.local_params:
            p.grad = None

    @contextlib.contextmanager
    def no_sync(self):
        """Skip gradient reduction (gradient-accumulation micro-steps)."""
        prev = self._sync_enabled
        self._sync_enabled = False
        try:
            yield
        finally:
            self._sync_enabled = prev
            for b in self.buckets:       # what was made so far, in place
                self._collect(b)

    @property
    def grad_scale(self) -> float:
        """1/world — folded into the fused AdamW step (SUM + pre-scale)."""
        return 1.0 / max(1, self.comm.world_size)

    def bucket_sizes_mb(self) -> List[float]:
        return [b.nbytes / (1 << 20) for b in self.buckets]
