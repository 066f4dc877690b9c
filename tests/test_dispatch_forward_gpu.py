"""fmoe_permute's paths against the C oracle, exactly: the one launch up to 4096 slots, the ranking
and placing kernels up to 64 or 256 ranking blocks (one pass or two over the expert columns) and the scan
beyond them."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import fastmoe_amd
from oracle import cref
from tests.helpers import to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,k,E,D,dtype,opts", [
    (1, 1, 1, 1, torch.bfloat16, {}),
    (1, 8, 256, 7168, torch.bfloat16, {}),
    (5, 3, 4, 100, torch.float16, {"int32": True}),           # 4-byte copies
    (31, 4, 4096, 7, torch.bfloat16, {"bad": True}),          # 2-byte copies, most experts empty
    (512, 8, 256, 264, torch.float32, {"strided": True}),     # 4096 slots: the last one-launch size
    (2048, 2, 3, 64, torch.bfloat16, {"bad": True}),
    (4097, 1, 5, 64, torch.bfloat16, {}),                     # one slot more
    (1024, 5, 1023, 72, torch.bfloat16, {"bad": True}),       # placed, one pass over the columns
    (1024, 5, 1024, 72, torch.float32, {"bad": True}),        # two passes
    (1024, 5, 1025, 72, torch.bfloat16, {}),                  # 256-slot ranking blocks: scan + fill
    (16384, 4, 37, 8, torch.bfloat16, {"int32": True}),       # 64 ranking blocks
    (13108, 5, 37, 4, torch.bfloat16, {}),                    # 65 of few experts: scan + fill
    (65536, 4, 128, 8, torch.bfloat16, {}),                   # 256 ranking blocks
    (52429, 5, 128, 4, torch.bfloat16, {}),                   # 257: scan + fill
    (4099, 2, 16, 1001, torch.bfloat16, {}),
])
def test_permutation_matches_the_oracle(T, k, E, D, dtype, opts):
    gen = torch.Generator().manual_seed(T + k + E)
    ids = torch.randint(0, E, (T, k), generator=gen)
    if opts.get("bad"):
        ids.view(-1)[::7] = E + 2
        ids.view(-1)[3::11] = -1
    if opts.get("int32"):
        ids = ids.int()
    gates = torch.rand(T, k, generator=gen)
    x = torch.randn(T, D + 8, generator=gen).to(dtype)
    xd = x.to(DEV)[:, :D]
    if not opts.get("strided"):
        xd = xd.contiguous()
    p = fastmoe_amd.permute_tokens(xd, ids.to(DEV), gates.to(DEV), E)
    counts, offsets, rev, slot_pos, _ = cref.permute(ids.long().numpy(), E)
    assert np.array_equal(p.expert_counts.cpu().numpy(), counts)
    assert np.array_equal(p.expert_offsets.cpu().numpy(), offsets)
    assert np.array_equal(p.reverse_map_indices.cpu().numpy(), rev)
    assert np.array_equal(p.slot_pos.cpu().numpy(), slot_pos)
    want = np.empty(T * k, np.float32)
    want[slot_pos] = gates.view(-1).numpy()
    assert np.array_equal(p.sorted_weights.cpu().numpy(), want)
    assert np.array_equal(to_np(p.permuted_data), to_np(x[:, :D])[rev])
    if opts.get("bad"):
        with pytest.raises(IndexError):
            fastmoe_amd.permute_tokens(xd, ids.to(DEV), gates.to(DEV), E, validate=True)
