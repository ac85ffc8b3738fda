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
    # bit for bit: 64 chains of every 64th exponential, a 32/16/8/4/2/1 butterfly,
    # an IEEE division (the exponential itself is the device's)
    maxima = np.array([scores[b:e].max(initial=-np.inf) for b, e in zip(crow, crow[1:])], dtype=np.float32)
    exps = torch.exp(torch.from_numpy(scores - np.repeat(maxima, lengths)).cuda()).cpu().numpy()
    want = np.empty_like(scores)
    for row, (b, e) in enumerate(zip(crow, crow[1:])):
        chains = np.zeros((-(-(e - b) // 64), 64), dtype=np.float32)
        chains.reshape(-1)[: e - b] = exps[b:e]
        d = np.zeros(64, dtype=np.float32)
        for step in chains:
            d = d + step
        for o in (32, 16, 8, 4, 2, 1):
            d = d + d[np.arange(64) ^ o]
        want[b:e] = exps[b:e] / d[0] if e > b else 0
    assert bitwise_equal(got, want)
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
