"""The atomic forward's few-tokens kernel (rows ordered by token within a workgroup): within the
bound of a reordered fp32 sum of the C oracle's result, at the edges of its tokens, slices and
shares."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import fastmoe_amd
from fastmoe_amd import _abi
from tests.helpers import abs_sum, oracle_fwd, reorder_tol, to_np, within_one_ulp16

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,counts,D,dtype,groups,opts", [
    (1, [1, 3], 1, torch.float32, 1, {}),
    (1, [9000], 65, torch.float32, 254, {}),                     # one token, 2 slices x 127 shares
    (16, [30, 0, 33], 64, torch.bfloat16, 1, {"bad": True}),     # 63 rows
    (16, [31, 0, 33], 64, torch.bfloat16, 1, {"bad": True}),     # 64
    (128, [5000, 3192, 1], 100, torch.float32, 32, {"int32": True}),  # shares end inside an expert
    (1024, [4096], 200, torch.float32, 4, {}),                   # the most tokens
    (1025, [4100], 200, torch.float32, 0, {}),                   # one more: k_fwd_atomic
    (1024, [8191], 8, torch.float32, 1, {}),                     # one share, a row short of full
    (7, [16385], 130, torch.float16, 255, {"w16": True}),        # 3 slices x 85 shares
    (3, [40, 80], 16400, torch.bfloat16, 257, {}),               # more slices than workgroups aimed at
    (3, [8000, 192], 8257, torch.bfloat16, 130, {}),             # one share of 8192 rows: a full list
    (3, [8000, 193], 8257, torch.bfloat16, 260, {}),             # one row more: two shares
])
@pytest.mark.parametrize("accumulate", [False, True])
def test_few_tokens_match_the_oracle(T, counts, D, dtype, groups, opts, accumulate, kernel_options):
    kernel_options(fwd_atomic_few=2)  # whatever the size rule says
    assert _abi.lib().fmoe_combine_atomic_few_groups(sum(counts), T, D) == groups
    gen = torch.Generator().manual_seed(T + D)
    experts = [torch.randn(n, D, generator=gen).to(dtype) for n in counts]
    N = sum(counts)
    idx = torch.randint(0, T, (N,), generator=gen)
    if opts.get("bad"):
        idx[::5] = T + 1
        idx[1::9] = -2
    w = torch.rand(N, generator=gen)
    if opts.get("w16"):
        w = w.to(dtype)
    wd, xd = w.to(DEV), [x.to(DEV) for x in experts]
    idxd = (idx.int() if opts.get("int32") else idx).to(DEV)
    init = torch.randn(T, D, generator=gen).to(dtype) if accumulate else None
    if accumulate:
        got = init.to(DEV)
        fastmoe_amd.grouped_weighted_scatter_add(xd, idxd, wd, (T, D), out=got, mode="atomic")
        acc0 = init.float().numpy()
    else:
        got = fastmoe_amd.grouped_weighted_scatter_add(xd, idxd, wd, (T, D), mode="atomic")
        acc0 = None
    want, acc, _ = oracle_fwd(experts, idx, w, T, dtype, acc_init=acc0)
    scale = abs_sum(experts, idx, w, T) + (np.abs(init.float().numpy()) if accumulate else 0.0)
    valid = idx[(idx >= 0) & (idx < T)]
    n = int(torch.bincount(valid, minlength=T).max()) + 1
    if dtype == torch.float32:
        assert np.all(np.abs(to_np(got).astype(np.float64) - acc) <= reorder_tol(n, scale))
    else:
        g = got.float().cpu().numpy()
        wantf = torch.from_numpy(want.view(np.int16)).view(dtype).float().numpy()
        assert np.all(within_one_ulp16(g, wantf, dtype, n, scale))


@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_indices_that_change_during_the_call_lose_no_row(dtype):
    """Another stream keeps swapping the indices between two valid routings: which of the two a row
    takes is open, but each row is added exactly once (rows of ones, unit gates: every column sums
    to N, which fp32 holds exactly)."""
    T, N, D = 128, 65536, 64
    assert _abi.lib().fmoe_combine_atomic_few_groups(N, T, D) == 128
    routes = [torch.full((N,), t, dtype=dtype, device=DEV) for t in (0, T - 1)]
    idx = routes[0].clone()
    x, w = torch.ones(N, D, device=DEV), torch.ones(N, device=DEV)
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    outs = []
    for i in range(20):
        with torch.cuda.stream(other):
            for j in range(8):
                idx.copy_(routes[(i + j) % 2])
        outs.append(fastmoe_amd.weighted_scatter_add(x, idx, w, (T, D), mode="atomic"))
    torch.cuda.synchronize()
    for out in outs:
        assert bool((out.sum(0) == N).all()) and not bool(out[1:T - 1].any())
