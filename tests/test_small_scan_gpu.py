"""The small forward's 256-id steps: windows that refill within a step, row counts around a step,
tokens of more rows than a step, and the sizes that the default choice now sends here -- equal to the
planned path bit for bit."""
from __future__ import annotations

import pytest
import torch

from fastmoe_amd import _abi, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,N,D,hot,dtype", [
    (1, 1, 8, 0.0, torch.bfloat16),
    (3, 255, 264, 0.0, torch.float32),
    (3, 256, 264, 0.5, torch.bfloat16),
    (3, 257, 264, 1.0, torch.bfloat16),      # 257 rows of one token
    (2, 4096, 64, 0.9, torch.float32),       # every step fills the window
    (5, 4095, 100, 0.3, torch.float16),
    (1024, 4096, 1024, 0.0, torch.bfloat16),  # T * N = 2^22
    (4096, 1024, 264, 0.1, torch.bfloat16),
])
@pytest.mark.parametrize("accumulate", [False, True])
def test_small_forward_equals_the_planned_one(T, N, D, hot, dtype, accumulate, kernel_options):
    gen = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(N, D, generator=gen, device=DEV).to(dtype)
    experts = [x[:N // 3], x[N // 3:N // 3], x[N // 3:]]
    idx = torch.randint(0, T, (N,), generator=gen, device=DEV)
    idx[torch.rand(N, generator=gen, device=DEV) < hot] = T // 2
    if N > 20:
        idx[::13] = T + 5
        idx[5::17] = -1
    w = torch.rand(N, generator=gen, device=DEV)
    init = torch.randn(T, D, generator=gen, device=DEV).to(dtype)
    outs = []
    for small in (2, 1):
        kernel_options(small=small)
        if accumulate:
            out = init.clone()
            ops.grouped_weighted_scatter_add(experts, idx, w, (T, D), out=out)
        else:
            out = ops.grouped_weighted_scatter_add(experts, idx, w, (T, D))
        outs.append(out)
    assert torch.equal(*outs)


def test_default_choice():
    assert ops._use_small(4096, 1024, 256) and not ops._use_small(4096, 1025, 256)
    assert ops._use_small(1024, 4096, 8) and not ops._use_small(512, 4097, 8)
    assert ops._use_small(8, 1 << 14, 8)  # T * N = 2^17, whatever T
    assert ops._use_small(2048, 256, 8, 32 << 20) and not ops._use_small(2048, 256, 8, (32 << 20) + 1)
    assert ops._use_small(1024, 128, 8, 1 << 30)
    assert _abi.option("small") == 0
