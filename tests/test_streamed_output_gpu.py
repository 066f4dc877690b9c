"""The deterministic forward's non-temporal output stores: outputs of 96 MiB or more that the call
overwrites, in a step or from 7 rows per token.  Sizes on both sides of that line, vector and element-wise columns, padded rows and an
accumulating call (which never takes them), bit for bit against the C oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from fastmoe_amd import _abi, ops
from tests.helpers import bits, oracle_fwd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,D,dtype,pad,accumulate", [
    (12287, 4096, torch.bfloat16, 0, False),   # one row below the line
    (12288, 4096, torch.bfloat16, 0, False),
    (12288, 4096, torch.bfloat16, 8, False),   # padded output rows
    (12288, 4096, torch.bfloat16, 0, True),
    (12300, 4097, torch.float16, 0, False),    # element-wise columns, a partial last chunk
    (6145, 4104, torch.float32, 0, False),     # vectors, a partial last chunk
])
@pytest.mark.parametrize("mode", [_abi.MODE_DET_STEP, _abi.MODE_DET])  # streamed, not
def test_large_outputs_match_the_oracle(T, D, dtype, pad, accumulate, mode):
    gen = torch.Generator().manual_seed(5)
    counts = [120, 0, 77, 103]
    experts = [torch.randn(n, D, generator=gen).to(dtype) for n in counts]
    N = sum(counts)
    idx = torch.randint(0, T, (N,), generator=gen)
    idx[:8] = T - 1  # a token of several rows in the last output row
    w = torch.rand(N, generator=gen)
    want, _, _ = oracle_fwd(experts, idx, w, T, dtype)
    meta, plan = ops.prepare_metadata_and_plan([x.to(DEV) for x in experts], idx.to(DEV),
                                               w.to(DEV), T)
    full = torch.full((T, D + pad), 0.0 if accumulate else 7.0, dtype=dtype, device=DEV)
    out = full[:, :D]
    ops._launch_fwd(meta, mode, plan, None, None, out, accumulate=accumulate)
    assert np.array_equal(bits(out), want.view(np.uint32) if dtype == torch.float32 else want)
    if pad:
        assert bool((full[:, D:] == 7.0).all())


@pytest.mark.parametrize("rows", [7, 6])  # per token: streamed by the forward alone, not
def test_forward_alone_and_in_a_step_agree(rows):
    T, D = 12288, 4096
    gen = torch.Generator(device=DEV).manual_seed(6)
    x = torch.randn(T * rows, D, generator=gen, device=DEV).bfloat16()
    idx = torch.randint(0, T, (T * rows,), generator=gen, device=DEV)
    w = torch.rand(T * rows, generator=gen, device=DEV)
    alone = ops.weighted_scatter_add(x, idx, w, (T, D))
    step = ops.weighted_scatter_add(x, idx, w.clone().requires_grad_(True), (T, D))
    assert step.requires_grad and torch.equal(alone, step.detach())
