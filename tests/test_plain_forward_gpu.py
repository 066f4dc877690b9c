"""A forward that records nothing gives what the recorded one gives, bit for bit: every mode, the
permutation, the slot-map combine, experts given as any iterable, and out-of-range checks."""
from __future__ import annotations

import pytest
import torch

import fastmoe_amd
from fastmoe_amd.workloads import Workload, make_experts, make_routing, make_topk

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("small", [2, 1])  # the one-launch small path, the planned path
@pytest.mark.parametrize("kind", ["no_grad", "inference", "no tensor requires grad"])
def test_combine_equals_the_recorded_forward(small, kind, kernel_options, library_calls):
    kernel_options(small=small)
    wl = Workload("t", 700, 264, 8, 4, torch.bfloat16, 3, False)
    idx, w, counts = make_routing(wl)
    xs = [x.to(DEV) for x in make_experts(counts, wl.D, wl.dtype, "cpu", 3)]
    idx, w = idx.to(DEV), w.to(DEV)
    T = wl.T
    shape = (T, wl.D)
    forward = "fmoe_combine_fwd_small" if small == 2 else "fmoe_combine_fwd"
    want = fastmoe_amd.grouped_weighted_scatter_add(xs, idx, w.clone().requires_grad_(True), shape)
    assert want.requires_grad and library_calls.pop() == forward
    if kind == "no_grad":
        with torch.no_grad():
            got = fastmoe_amd.grouped_weighted_scatter_add(
                [x.requires_grad_(True) for x in xs], idx, w, shape)
    elif kind == "inference":
        with torch.inference_mode():
            got = fastmoe_amd.grouped_weighted_scatter_add(xs, idx, w, shape)
            assert got.is_inference()
    else:
        got = fastmoe_amd.grouped_weighted_scatter_add((x for x in xs), idx, w, shape)
    assert not got.requires_grad and got.grad_fn is None and library_calls[-1] == forward
    assert torch.equal(got, want.detach())
    with torch.no_grad(), pytest.raises(IndexError):
        fastmoe_amd.grouped_weighted_scatter_add(xs, idx + T, w, shape, validate=True)
    atomic = fastmoe_amd.grouped_weighted_scatter_add(xs, idx, w, shape, mode="atomic")
    torch.testing.assert_close(atomic.float(), want.detach().float(), rtol=2 ** -7, atol=2 ** -7)


@pytest.mark.parametrize("small", [1, 2])  # the slot-map plan, the small path
def test_layer_stages_equal_the_recorded_ones(small, kernel_options, library_calls):
    kernel_options(small=small)
    wl = Workload("t", 600, 264, 8, 4, torch.float32, 4, False)
    ids, gates = (t.to(DEV) for t in make_topk(wl))
    x = torch.randn(wl.T, wl.D, generator=torch.Generator().manual_seed(1)).to(DEV)
    rec = fastmoe_amd.permute_tokens(x.clone().requires_grad_(True), ids, gates, wl.E)
    p = fastmoe_amd.permute_tokens(x, ids, gates, wl.E)
    for a, b in zip(p, rec):
        assert torch.equal(a, b) and not a.requires_grad
    parts = list(p.permuted_data.split(p.expert_counts.tolist()))
    outs = []
    for w in (p.sorted_weights, p.sorted_weights.clone().requires_grad_(True)):
        outs.append(fastmoe_amd.unpermute(parts, p.reverse_map_indices, w, (1, wl.T),
                                          permutation=p))
    assert torch.equal(outs[0], outs[1].detach()) and not outs[0].requires_grad
    plans = library_calls.count("fmoe_build_metadata_and_plan_from_slots")
    assert plans == (2 if small == 1 else 0)
