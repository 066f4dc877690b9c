"""When a call may run its forward without the autograd Function: only when nothing is recorded and
nothing else watches the call (grad mode, requires_grad of any tensor, functorch, forward mode,
tracing, compilation, tensors that escaped from a finished transform)."""
from __future__ import annotations

import pytest
import torch
from torch.autograd import forward_ad

import fastmoe_amd
from fastmoe_amd import _host, dispatch, moe, ops


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


def _escaped(x, transform):
    """``x`` as a finished torch.func transform left it to the caller: still a wrapper, its level
    dead."""
    seen = []

    def f(z, *_):
        y = x.view_as(x) + 0 * z.to(x.dtype)
        seen.append(y)
        return z.sum()

    z = torch.zeros(())
    torch.func.grad(f)(z) if transform == "grad" else torch.func.jvp(f, (z,), (z,))
    assert torch._C._functorch.is_functorch_wrapped_tensor(seen[0])
    return seen[0]


@pytest.mark.parametrize("transform", ["grad", "jvp"])
def test_escaped_wrappers_keep_the_function(transform):
    """Function.apply hands its forward the tensor inside a dead wrapper, which has the data that the
    wrapper itself cannot show; any argument may be one, the indices too."""
    t = _escaped(torch.zeros(2, 3), transform)
    assert _host.wrapped([torch.zeros(1), t]) and not _host.wrapped([*_tensors(), None, 3])
    with torch.no_grad():
        assert not ops._runs_plain((torch.zeros(2), t))
        with pytest.raises(TypeError):
            _host.wrapped(7)


@pytest.mark.parametrize("transform", ["grad", "jvp"])
@pytest.mark.parametrize("at", ["expert", "gates", "indices"])
def test_combine_and_layer_take_escaped_wrappers(transform, at, monkeypatch):
    got = []

    def forward(ctx, mode, validate, indices, weights, out_shape, experts, w_grad, slots=None):
        got.append([t.data_ptr() for t in (indices, weights, *experts)])  # the data is there
        return torch.zeros(out_shape)

    for module in (ops, moe):
        monkeypatch.setattr(module, "_combine_forward", forward)
    monkeypatch.setattr(ops, "_require_cuda", lambda t, what: None)
    t = {"expert": torch.zeros(4, 3), "gates": torch.zeros(4),
         "indices": torch.zeros(4, dtype=torch.long)}
    t[at] = _escaped(t[at], transform)
    with torch.no_grad():
        fastmoe_amd.grouped_weighted_scatter_add([t["expert"]], t["indices"], t["gates"], (2, 3))
        p = fastmoe_amd.PermutedTokens(*[None] * 5, slot_pos=torch.zeros(4, dtype=torch.int32))
        fastmoe_amd.unpermute([t["expert"]], t["indices"], t["gates"], (1, 2), permutation=p)
    assert len(got) == 2


@pytest.mark.parametrize("transform", ["grad", "jvp"])
@pytest.mark.parametrize("at", ["x", "ids", "gates"])
def test_dispatch_takes_escaped_wrappers(transform, at, monkeypatch):
    def permute(x, gates, ids, num_experts, validate):
        assert x.data_ptr() and gates.data_ptr() and ids.data_ptr()
        return (x.clone(), gates.reshape(-1).clone(), *(torch.zeros(4, dtype=torch.long)
                                                        for _ in range(4)))

    monkeypatch.setattr(dispatch, "_permute", permute)
    monkeypatch.setattr(dispatch, "_require_cuda", lambda t, what: None)
    t = {"x": torch.zeros(2, 3), "ids": torch.zeros(2, 2, dtype=torch.long),
         "gates": torch.zeros(2, 2)}
    t[at] = _escaped(t[at], transform)
    with torch.no_grad():
        p = fastmoe_amd.permute_tokens(t["x"], t["ids"], t["gates"], 4)
    assert p.permuted_data.shape == (2, 3)
