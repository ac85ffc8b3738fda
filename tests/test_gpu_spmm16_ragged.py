"""16-bit SpMM, rows whole, on widths whose last 16-byte lane overlaps the one
before: every lane count and feature tile, odd widths (2-byte aligned rows) and
unaligned X, bit for bit the oracle's fp64 sums, rounded."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from autosage_amd import _native
from gpu_common import case_graph, require_gpu, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("features", [7, 8, 9, 15, 33, 47, 63, 64, 65, 100, 127, 129, 255, 257, 259, 511, 513])
def test_ragged_widths(features, weighted, dtype):
    crow, col = case_graph(500, 11, seed=features, hubs=2, hub_degree=400, empty=0.1)
    rng = np.random.default_rng(features)
    # small integers: every order of the additions is exact
    x = torch.from_numpy(rng.integers(-8, 9, (500, features)).astype(np.float32)).to(dtype)
    val = torch.from_numpy(rng.integers(-3, 4, col.size).astype(np.float32)).to(dtype) if weighted else None
    want = oracle.spmm_rounded_16(crow, col, val, x, dtype).view(torch.int16)
    d = to_dev(crow, col)
    d_val = None if val is None else val.cuda()
    flat = torch.empty(x.numel() + 1, dtype=dtype, device="cuda")
    flat[1:] = x.reshape(-1).cuda()
    for d_x in (x.cuda(), flat[1:].view(x.shape)):
        assert torch.equal(_native.spmm_rows_16_impl(*d, d_val, d_x).cpu().view(torch.int16), want)
