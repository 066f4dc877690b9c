"""The deterministic forward's non-temporal output stores: outputs of 96 MiB or more that the call
overwrites.  Sizes on both sides of that line, vector and element-wise columns, padded rows and an
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
def test_large_outputs_match_the_oracle(T, D, dtype, pad, accumulate):
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
    ops._launch_fwd(meta, _abi.MODE_DET, plan, None, None, out, accumulate=accumulate)
    assert np.array_equal(bits(out), want.view(np.uint32) if dtype == torch.float32 else want)
    if pad:
        assert bool((full[:, D:] == 7.0).all())
