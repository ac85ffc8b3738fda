"""16-bit SDDMM by blocks of edges on rows whose last 16-byte chunk is read
at F - 8: every lane count, every overlap, odd widths (2-byte aligned rows) and
unaligned views, bit for bit the oracle's fp64 sums, rounded."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from gpu_common import case_graph, require_gpu, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def _unaligned(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    flat[1:] = t.reshape(-1).cuda()
    return flat[1:].view(t.shape)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("features", [8, 9, 10, 11, 15, 17, 31, 33, 47, 63, 65, 68, 100, 127, 129, 199, 255, 257, 300, 511,
                                      512, 513])
def test_ragged_widths(features, dtype):
    crow, col = case_graph(700, 9, seed=features, hubs=2, hub_degree=600, empty=0.08)
    rng = np.random.default_rng(features)
    q, k = (torch.from_numpy(rng.standard_normal((700, features)).astype(np.float32)).to(dtype) for _ in range(2))
    # an infinity where the last chunk overlaps the one before counts once, and no 0 * inf
    k[5, max(features - 8, 0)] = float("inf")
    k[6, features - 1] = -float("inf")
    want = oracle.sddmm_rounded_16(crow, col, q, k, dtype).view(torch.int16)
    d = to_dev(crow, col)
    for d_q, d_k in ((q.cuda(), k.cuda()), (_unaligned(q), k.cuda()), (q.cuda(), _unaligned(k))):
        got = torch.ops.autosage.sddmm_csr(*d, d_q, d_k).cpu().view(torch.int16)
        assert torch.equal(got, want)
