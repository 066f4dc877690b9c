"""When a call may run its forward without the autograd Function: only when nothing is recorded and
nothing else watches the call (grad mode, requires_grad of any tensor, functorch, forward mode,
tracing, compilation)."""
from __future__ import annotations

import pytest
import torch
from torch.autograd import forward_ad

from fastmoe_amd import _host, ops


def _tensors(grad_at=None):
    return tuple(torch.zeros(2, 3, requires_grad=i == grad_at) for i in range(4))


def test_helper_looks_at_every_tensor():
    assert not _host.requires_grad(_tensors())
    for i in range(4):
        assert _host.requires_grad(_tensors(i))
    assert not _host.requires_grad([]) and not _host.requires_grad([None, 3])
    with pytest.raises(TypeError):
        _host.requires_grad(7)


def test_grad_mode_and_requires_grad_decide():
    assert ops._runs_plain(_tensors())
    assert not ops._runs_plain(_tensors(0)) and not ops._runs_plain(_tensors(3))
    with torch.no_grad():
        assert ops._runs_plain(_tensors(3))
    with torch.inference_mode():
        assert ops._runs_plain(_tensors())


def test_watchers_keep_the_function():
    seen = []

    def f(x):
        seen.append(ops._runs_plain((x,)))
        return x * 2

    with torch.no_grad():
        torch.func.vmap(f)(torch.zeros(3))
        torch.func.jvp(f, (torch.zeros(3),), (torch.ones(3),))
        with forward_ad.dual_level():
            f(torch.zeros(3))
        torch.jit.trace(f, torch.zeros(3), check_trace=False)
    assert seen == [False] * 4
