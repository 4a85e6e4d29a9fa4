"""A block's norms beside their residual: a norm that is more than its class's
forward is called as a module."""

import pytest
import torch

from scaffold.models.gpt2 import LayerNorm
from scaffold.models.llama import RMSNorm


@pytest.mark.parametrize("cls", [LayerNorm, RMSNorm])
@pytest.mark.parametrize("how", ["plain", "hook", "pre", "backward", "global",
                                 "subclass", "instance", "compiled"])
def test_norms_with_hooks_are_called(cls, how):
    calls = []
    norm = type("Other", (cls,), {"forward": lambda s, x: calls.append(1) or x})(8) \
        if how == "subclass" else cls(8)
    x = torch.randn(2, 8, requires_grad=True)
    handle = None
    if how == "hook":
        norm.register_forward_hook(lambda *a: calls.append(1))
    elif how == "pre":
        norm.register_forward_pre_hook(lambda *a: calls.append(1))
    elif how == "backward":
        norm.register_full_backward_hook(lambda *a: calls.append(1))
    elif how == "global":
        handle = torch.nn.modules.module.register_module_forward_hook(
            lambda *a: calls.append(1))
    elif how == "instance":
        norm.forward = lambda x: calls.append(1) or x
    elif how == "compiled":
        norm.compile(backend=lambda graph, _: calls.append(1) or graph.forward)
    try:
        y, same = cls.fork(norm, x)
        (y.sum() + same.sum()).backward()
    finally:
        if handle is not None:
            handle.remove()
    assert torch.equal(same, x) and len(calls) == (how != "plain")
    if how not in ("subclass", "instance"):
        assert torch.equal(y, cls.forward(norm, x))
