"""fmoe_permute's paths against the C oracle, exactly: the one launch up to 4096 slots, the ranking
and placing kernels up to 64 or 256 ranking blocks (one pass or two over the expert columns) and the scan
beyond them."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import fastmoe_amd
from fastmoe_amd import _abi
from oracle import cref
from tests.helpers import to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,k,E,D,dtype,opts", [
    (1, 1, 1, 1, torch.bfloat16, {}),
    (1, 8, 256, 7168, torch.bfloat16, {}),
    (1, 1, 4096, 64, torch.bfloat16, {}),                     # most workgroups only count experts
    (2, 8, 1023, 264, torch.bfloat16, {"bad": True}),
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


@pytest.mark.parametrize("T,k,E,bad", [(1, 1, 1, False), (37, 3, 8, True), (512, 8, 256, True),
                                       (300, 4, 3000, False), (1000, 4, 1024, True)])
def test_separate_calls_give_the_one_launch_outputs(T, k, E, bad):
    """fmoe_permute_build and fmoe_permute_gather at sizes that fmoe_permute takes in one launch."""
    gen = torch.Generator().manual_seed(T)
    ids = torch.randint(0, E, (T, k), generator=gen)
    if bad:
        ids.view(-1)[::5] = E
    ids, gates = ids.to(DEV), torch.rand(T, k, generator=gen).to(DEV)
    x = torch.randn(T, 40, generator=gen).to(DEV)
    p = fastmoe_amd.permute_tokens(x, ids, gates, E)
    lib, N, stream = _abi.lib(), T * k, torch.cuda.current_stream().cuda_stream
    got = [torch.full_like(t, 7) for t in p]
    rows, counts, rev, sorted_gates, offsets, slot_pos = got
    status = torch.empty(1, dtype=torch.int32, device=DEV)
    ws = torch.empty(lib.fmoe_permute_workspace_bytes(N, E), dtype=torch.uint8, device=DEV)
    _abi.check(lib.fmoe_permute_build(
        ids.data_ptr(), _abi.I64, gates.data_ptr(), _abi.F32, T, k, E, counts.data_ptr(),
        offsets.data_ptr(), rev.data_ptr(), sorted_gates.data_ptr(), slot_pos.data_ptr(),
        status.data_ptr(), ws.data_ptr(), stream), "fmoe_permute_build")
    _abi.check(lib.fmoe_permute_gather(slot_pos.data_ptr(), T, k, 160, x.data_ptr(), 160,
                                       rows.data_ptr(), stream), "fmoe_permute_gather")
    for a, b in zip(got, p):
        assert torch.equal(a, b)
    assert int(status) == (len(range(0, N, 5)) if bad else 0)


@pytest.mark.parametrize("E,block", [(1024, 1024), (1025, 256)])  # rank + place; rank + scan + fill
def test_ids_overwritten_after_ranking_write_nothing_outside(E, block):
    """The ids lie where the ranking kernel stores its ranks, so the kernel that places the slots
    reads the ranks as ids.  All ids are 0: slot i's rank r = i mod block is its new id, and for
    r > 0 expert r begins at row N, past the outputs.  Only r == 0 has a place; nothing else is
    written."""
    T, k = 1024, 3
    N, guard = T * k, 2048
    nb = N // block
    rank_at = (nb * (E + 1) * 4 + 255) // 256 * 256  # block counts first, then the ranks
    lib = _abi.lib()
    nbytes = lib.fmoe_permute_workspace_bytes(N, E)
    assert rank_at + N * 4 <= nbytes
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=DEV)  # ids: all 0
    gates = torch.rand(N, device=DEV)
    counts = torch.empty(E, dtype=torch.int64, device=DEV)
    offsets = torch.empty(E + 1, dtype=torch.int64, device=DEV)
    status = torch.empty(1, dtype=torch.int32, device=DEV)
    rev = torch.full((N + guard,), -7, dtype=torch.int64, device=DEV)
    sorted_gates = torch.full((N + guard,), -7.0, device=DEV)
    slot_pos = torch.full((N + guard,), -7, dtype=torch.int32, device=DEV)
    rc = lib.fmoe_permute_build(
        ws.data_ptr() + rank_at, _abi.I32, gates.data_ptr(), _abi.F32, T, k, E, counts.data_ptr(),
        offsets.data_ptr(), rev.data_ptr(), sorted_gates.data_ptr(), slot_pos.data_ptr(),
        status.data_ptr(), ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
    _abi.check(rc, "fmoe_permute_build")
    at = torch.arange(0, N, block, device=DEV)
    for got, want in ((rev, at // k), (sorted_gates, gates[at]), (slot_pos, at.int())):
        expect = torch.full_like(got, -7)
        expect[at] = want.to(got.dtype)
        assert torch.equal(got, expect)
    assert int(counts[0]) == N and int(status) == 0
