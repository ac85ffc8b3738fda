"""The row softmax and its backward where a row changes hands: 16 lanes and
1 to 4 slots, a wave (in registers or in steps of 512 edges), the workgroup."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from autosage_amd._native import csr_row_softmax_backward_impl
from gpu_common import bitwise_equal, require_gpu, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


LENGTHS = [0, 1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 127, 511, 512, 513, 1025, 4095, 4096, 4097, 6144, 6145,
           0, 20001, 5, 9000, 3]


@pytest.mark.parametrize("order", ["as listed", "shuffled", "reversed"])
def test_softmax_rows_of_every_length(order):
    rng = np.random.default_rng(11)
    lengths = np.array(LENGTHS)
    lengths = {"as listed": lengths, "shuffled": rng.permutation(lengths), "reversed": lengths[::-1]}[order]
    crow = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    scores = (rng.standard_normal(int(crow[-1])) * 3).astype(np.float32)
    # a masked edge (-inf) in a row of each kind
    for row in range(lengths.size):
        if lengths[row] > 1:
            scores[crow[row] + lengths[row] // 2] = -np.inf
    d_crow, d_scores = to_dev(crow, scores)
    got = torch.ops.autosage.csr_row_softmax(d_crow, d_scores)
    ref = oracle.row_softmax(crow, scores)
    assert np.all(np.abs(got.cpu().numpy() - ref) <= 1e-6 + 1e-5 * np.abs(ref))
    # the denominator's order: an attention over one-hot values computes the
    # same probabilities in one wave (or four) per row
    n = lengths.size
    q = rng.standard_normal((n, 32)).astype(np.float32)
    k = rng.standard_normal((n, 32)).astype(np.float32)
    v = rng.standard_normal((n, 8)).astype(np.float32)
    col = rng.integers(0, n, size=int(crow[-1])).astype(np.int64)
    d_col, d_q, d_k, d_v = to_dev(col, q, k, v)
    probs = torch.ops.autosage.csr_row_softmax(d_crow, torch.ops.autosage.sddmm_csr(d_crow, d_col, d_q, d_k))
    fused = torch.ops.autosage.csr_attention(d_crow, d_col, d_q, d_k, d_v, 1.0)
    assert torch.equal(torch.ops.autosage.spmm_csr(d_crow, d_col, probs, d_v), fused)
    grad = rng.standard_normal(scores.size).astype(np.float32)
    (d_grad,) = to_dev(grad)
    back = csr_row_softmax_backward_impl(d_crow, got, d_grad)
    assert bitwise_equal(back, oracle.row_softmax_backward(crow, got.cpu().numpy(), grad))


def test_softmax_rows_with_infinities_and_nan():
    """As with one wave per row: a row with +inf or NaN is NaN throughout, a row
    of -inf alone too, whatever its length; its neighbours are not touched."""
    lengths = np.array([3, 40, 3, 200, 3, 5000, 3, 700, 3])
    crow = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    for special in (np.inf, np.nan, -np.inf):
        scores = np.random.default_rng(5).standard_normal(int(crow[-1])).astype(np.float32)
        for row in (1, 3, 5, 7):
            if special == -np.inf:
                scores[crow[row]:crow[row + 1]] = special
            else:
                scores[crow[row] + lengths[row] - 1] = special
        got = torch.ops.autosage.csr_row_softmax(*to_dev(crow, scores)).cpu().numpy()
        for row in range(lengths.size):
            part = got[crow[row]:crow[row + 1]]
            assert np.all(np.isnan(part)) if row % 2 else abs(part.sum() - 1) < 1e-5
