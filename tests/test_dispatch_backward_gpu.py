"""The permutation's one-launch backward (fmoe_permute_backward) against the C oracle's combine with
unit gates, bit for bit: every tile, rows that no 16-byte vector divides, unaligned gradient rows, k
from 1 to 64 (and 65, which takes the planned combine), and each gradient asked for alone.  Sizes whose
grad_x is streamed or whose workgroups are bounded: against the planned combine."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import fastmoe_amd
from fastmoe_amd import _abi, dispatch
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


_CODES = {torch.float32: _abi.F32, torch.bfloat16: _abi.BF16, torch.float16: _abi.F16}


# tile: fmoe_combine_det_tile's <U><R>, 0 for element-wise rows, None for the planned combine
@pytest.mark.parametrize("T,k,E,D,dtype,gate_dtype,shift,tile", [
    (1, 1, 1, 1, torch.float32, torch.float32, 0, 0),
    (37, 1, 4, 4096, torch.bfloat16, torch.float32, 0, 42),   # one row per token
    (37, 2, 4, 1024, torch.bfloat16, torch.bfloat16, 0, 18),
    (37, 2, 4, 2048, torch.float16, torch.float32, 0, 24),
    (37, 2, 4, 4096, torch.bfloat16, torch.float32, 0, 44),
    (37, 6, 8, 4096, torch.bfloat16, torch.float32, 0, 24),   # few wave units
    (37, 4, 8, 2048, torch.bfloat16, torch.float32, 0, 28),
    (37, 8, 8, 7168, torch.float16, torch.float16, 0, 18),
    (640, 4, 8, 4096, torch.bfloat16, torch.bfloat16, 0, 42),  # 1280 wave units
    (512, 4, 8, 1536, torch.bfloat16, torch.float32, 0, 24),   # 1024 of 2 vectors
    (37, 4, 8, 1032, torch.float32, torch.float32, 0, 28),    # a partial last chunk
    (37, 5, 8, 1001, torch.float16, torch.float16, 0, 0),     # element-wise
    (37, 5, 8, 1024, torch.bfloat16, torch.float32, 3, 18),   # gradient rows off 16 bytes: element-wise
    (5, 64, 80, 264, torch.bfloat16, torch.float32, 0, 18),
    (5, 65, 80, 264, torch.bfloat16, torch.float32, 0, None),  # planned combine
])
def test_backward_matches_the_oracle(T, k, E, D, dtype, gate_dtype, shift, tile, library_calls):
    if tile is not None:
        assert _abi.lib().fmoe_combine_det_tile(T * k, T, D, _CODES[dtype]) == tile
    x, ids, gates, g_rows, g_gates = _inputs(T, k, E, D, dtype, gate_dtype)
    xd = x.to(DEV).requires_grad_(True)
    gd = gates.to(DEV).requires_grad_(True)
    p = fastmoe_amd.permute_tokens(xd, ids.to(DEV), gd, E)
    flat = torch.empty(g_rows.numel() + shift, dtype=dtype, device=DEV)
    rows = flat[shift:].view(g_rows.shape).copy_(g_rows)
    gx, gg = torch.autograd.grad([p.permuted_data, p.sorted_weights], [xd, gd],
                                 [rows, g_gates.to(DEV)])
    assert ("fmoe_permute_backward" in library_calls) == (tile is not None)
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


@pytest.mark.parametrize("T,k,D,dtype,tile", [
    (6144, 2, 4096, torch.bfloat16, 44),     # grad_x of 48 MiB: streamed
    (6143, 2, 4096, torch.bfloat16, 44),     # a row less: not
    (6150, 1, 4097, torch.float16, 0),       # streamed, element-wise
    (8192, 4, 4096, torch.bfloat16, 324),    # rows of 256 MiB: 3 workgroups to a CU, streamed
    (5462, 3, 8192, torch.bfloat16, 424),    # 3 rows per token: 4
    (4100, 8, 12288, torch.bfloat16, 224),   # 769 MiB: 2
    (2050, 8, 8200, torch.float32, 324),     # fp32, a partial last chunk
])
def test_large_backward_equals_the_planned_combine(T, k, D, dtype, tile, kernel_options):
    assert _abi.lib().fmoe_combine_det_tile(T * k, T, D, _CODES[dtype]) == tile
    gen = torch.Generator(device=DEV).manual_seed(2)
    ids = torch.randint(0, 64, (T, k), generator=gen, device=DEV)
    gates = torch.rand(T, k, generator=gen, device=DEV).requires_grad_(True)
    x = torch.zeros(T, D, dtype=dtype, device=DEV, requires_grad=True)
    p = fastmoe_amd.permute_tokens(x, ids, gates, 64)
    rows = torch.randn(T * k, D, generator=gen, device=DEV).to(dtype)
    g_gates = torch.rand(T * k, generator=gen, device=DEV)
    gx, gg = torch.autograd.grad([p.permuted_data, p.sorted_weights], [x, gates], [rows, g_gates])
    assert torch.equal(gg.view(-1), g_gates[p.slot_pos.long()])
    kernel_options(fwd_tile=44, small=1)
    assert torch.equal(gx, dispatch._unit_gate_combine(rows, p.reverse_map_indices, T))
