"""The deterministic forward's choice of tile and resident workgroups: every branch of the rule gives
what a fixed tile gives, bit for bit, with and without an output to accumulate into (the fixed tile
itself is held to the oracle elsewhere)."""
from __future__ import annotations

import pytest
import torch

from fastmoe_amd import _abi, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,D,N,dtype", [
    (512, 2048, 4096, torch.bfloat16),       # few wave units: the tile by D and r
    (639, 4096, 2556, torch.bfloat16),       # 1278 of 4 vectors: still
    (640, 4096, 2560, torch.bfloat16),       # 1280
    (511, 1536, 2044, torch.bfloat16),       # 1022 of 2 vectors
    (512, 2048, 768, torch.bfloat16),        # r = 1.5
    (512, 2048, 1279, torch.bfloat16),       # below 2.5
    (512, 2056, 1280, torch.bfloat16),       # 2.5, small rows
    (512, 1000, 2048, torch.bfloat16),       # less than a chunk of 2 vectors per lane
    (512, 1536, 2048, torch.bfloat16),       # less than a chunk of 4
    (512, 4104, 2048, torch.float16),        # a partial last chunk
    (4097, 8192, 16384, torch.bfloat16),     # 256 MiB, r just below 4: 3 workgroups
    (4681, 8192, 16383, torch.bfloat16),     # one row below 256 MiB
    (5462, 8192, 16384, torch.bfloat16),     # 256 MiB, r = 3: 4 workgroups
    (2048, 12288, 32768, torch.bfloat16),    # 768 MiB, r = 16: 2 workgroups
    (4682, 6144, 32768, torch.float32),      # 768 MiB, r just below 7
    (4681, 6148, 32768, torch.float32),      # just above both, a partial last chunk
])
@pytest.mark.parametrize("accumulate", [False, True])
def test_every_branch_equals_a_fixed_tile(T, D, N, dtype, accumulate, kernel_options):
    gen = torch.Generator(device=DEV).manual_seed(11)
    x = torch.randn(N, D, generator=gen, device=DEV).to(dtype)
    idx = torch.randint(0, T, (N,), generator=gen, device=DEV)
    w = torch.rand(N, generator=gen, device=DEV)
    init = torch.randn(T, D, generator=gen, device=DEV).to(dtype)
    meta, plan = ops.prepare_metadata_and_plan([x], idx, w, T)
    outs = []
    for tile in (0, 44):
        kernel_options(fwd_tile=tile)
        out = init.clone()
        ops._launch_fwd(meta, _abi.MODE_DET, plan, None, None, out, accumulate=accumulate)
        outs.append(out)
    assert torch.equal(*outs)
