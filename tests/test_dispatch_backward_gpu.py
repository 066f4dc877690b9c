"""The permutation's one-launch backward (fmoe_permute_backward) against the C oracle's combine with
unit gates, bit for bit: every tile choice, rows that no 16-byte vector divides, unaligned gradient
rows, k from 1 to 64 (and 65, which takes the planned combine), and each gradient asked for alone."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import fastmoe_amd
from tests.helpers import bits, oracle_fwd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(T, k, E, D, dtype, gate_dtype, seed=3):
    gen = torch.Generator().manual_seed(seed)
    ids = torch.stack([torch.randperm(max(E, k), generator=gen)[:k] % E for _ in range(T)])
    return (torch.randn(T, D, generator=gen).to(dtype), ids,
            torch.rand(T, k, generator=gen).to(gate_dtype),
            torch.randn(T * k, D, generator=gen).to(dtype),
            torch.randn(T * k, generator=gen).to(gate_dtype))


def _want(p, ids, g_rows, g_gates, T):
    rev = p.reverse_map_indices.cpu()
    gx, _, _ = oracle_fwd([g_rows], rev, torch.ones(rev.numel()), T, g_rows.dtype)
    gg = g_gates[p.slot_pos.cpu().long()].view(ids.shape)
    return (gx.view(np.uint32) if gx.dtype == np.float32 else gx), bits(gg)


@pytest.mark.parametrize("T,k,E,D,dtype,gate_dtype,shift", [
    (1, 1, 1, 1, torch.float32, torch.float32, 0),
    (37, 1, 4, 4096, torch.bfloat16, torch.float32, 0),      # one row per token: 4 x 2 tile
    (37, 2, 4, 1024, torch.bfloat16, torch.bfloat16, 0),     # 2 x 4
    (37, 6, 8, 4096, torch.bfloat16, torch.float32, 0),      # 4 x 4
    (37, 8, 8, 7168, torch.float16, torch.float16, 0),       # 1 x 8
    (37, 4, 8, 1032, torch.float32, torch.float32, 0),       # a partial last chunk
    (37, 5, 8, 1001, torch.float16, torch.float16, 0),       # element-wise
    (37, 5, 8, 1024, torch.bfloat16, torch.float32, 3),      # gradient rows off 16 bytes
    (5, 64, 80, 264, torch.bfloat16, torch.float32, 0),
    (5, 65, 80, 264, torch.bfloat16, torch.float32, 0),      # planned combine
])
def test_backward_matches_the_oracle(T, k, E, D, dtype, gate_dtype, shift):
    x, ids, gates, g_rows, g_gates = _inputs(T, k, E, D, dtype, gate_dtype)
    xd = x.to(DEV).requires_grad_(True)
    gd = gates.to(DEV).requires_grad_(True)
    p = fastmoe_amd.permute_tokens(xd, ids.to(DEV), gd, E)
    flat = torch.empty(g_rows.numel() + shift, dtype=dtype, device=DEV)
    rows = flat[shift:].view(g_rows.shape).copy_(g_rows)
    gx, gg = torch.autograd.grad([p.permuted_data, p.sorted_weights], [xd, gd],
                                 [rows, g_gates.to(DEV)])
    want_gx, want_gg = _want(p, ids, g_rows, g_gates, T)
    assert np.array_equal(bits(gx), want_gx)
    assert np.array_equal(bits(gg), want_gg)


def test_each_gradient_alone():
    """An output that the loss does not use has no gradient: the input it comes from gets zeros."""
    x, ids, gates, g_rows, g_gates = _inputs(19, 3, 5, 256, torch.float32, torch.float32)
    xd, gd = x.to(DEV).requires_grad_(True), gates.to(DEV).requires_grad_(True)
    p = fastmoe_amd.permute_tokens(xd, ids.to(DEV), gd, 5)
    want_gx, want_gg = _want(p, ids, g_rows, g_gates, 19)
    gx, gg = torch.autograd.grad(p.permuted_data, [xd, gd], g_rows.to(DEV), retain_graph=True)
    assert np.array_equal(bits(gx), want_gx) and not gg.any()
    gx, gg = torch.autograd.grad(p.sorted_weights, [xd, gd], g_gates.to(DEV))
    assert np.array_equal(bits(gg), want_gg) and not gx.any()
    p = fastmoe_amd.permute_tokens(x.to(DEV), ids.to(DEV), gd, 5)  # only the gates need one
    gg, = torch.autograd.grad(p.sorted_weights, [gd], g_gates.to(DEV))
    assert np.array_equal(bits(gg), want_gg)
