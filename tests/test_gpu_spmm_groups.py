"""The fp32 whole-graph SpMM in lane groups and workgroups on long rows, bit
for bit against the sequential product: widths around the lane and slice
bounds, rows around the batch, tile and long-row bounds, rows handed out
within a wave, one wave per row on graphs known to be even."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from autosage_amd import _native
from gpu_common import bitwise_equal, mismatch_report, require_gpu, to_dev

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 4, 5, 7, 8, 9, 16, 17, 255, 256, 257, 287, 288, 289, 383, 384, 385, 700, 768, 2305, 0, 3]


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def _graph(lengths, seed):
    rng = np.random.default_rng(seed)
    lengths = rng.permutation(np.asarray(lengths))
    crow = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    return crow, rng.integers(0, lengths.size, size=int(crow[-1])).astype(np.int64), rng


def _check(crow, col, val, x):
    ref = oracle.spmm_seq(crow, col, val, x)
    d_crow, d_col, d_x = to_dev(crow, col, x)
    d_val = None if val is None else to_dev(val)[0]
    got = torch.ops.autosage.spmm_csr(d_crow, d_col, d_val, d_x)
    assert bitwise_equal(got, ref), mismatch_report(got, ref)
    # X and Y 4 bytes off a vector's alignment, columns of unknown range
    off_x = torch.empty(d_x.numel() + 1, device="cuda")[1:].view_as(d_x).copy_(d_x)
    off_y = torch.full((d_x.numel() + 1,), float("nan"), device="cuda")[1:].view_as(d_x)
    status = _native.library().as_spmm_csr_f32(
        d_crow.data_ptr(), d_col.data_ptr(), None if d_val is None else d_val.data_ptr(), off_x.data_ptr(),
        off_y.data_ptr(), crow.size - 1, col.size, x.shape[1], 1, torch.cuda.current_stream().cuda_stream)
    assert status == 0
    torch.cuda.synchronize()
    assert bitwise_equal(off_y, ref), mismatch_report(off_y, ref)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("features", [3, 4, 5, 7, 8, 9, 12, 16, 17, 29, 32, 33, 47, 63, 64, 65, 69, 100, 128, 129, 200,
                                      256, 257, 300, 16641])
def test_spmm_groups_bitwise(features, weighted):
    lengths = LENGTHS * 3 if features < 1000 else LENGTHS[:11]
    crow, col, rng = _graph(lengths, features)
    x = rng.standard_normal((len(lengths), features)).astype(np.float32)
    val = rng.standard_normal(col.size).astype(np.float32) if weighted else None
    _check(crow, col, val, x)


def test_spmm_groups_leave_other_rows_alone():
    """Infinities of X reach the rows that gather them only, though absent
    edges of a batch and a row's overlapping lanes read X too."""
    crow, col, rng = _graph(LENGTHS, 3)
    x = rng.standard_normal((len(LENGTHS), 50)).astype(np.float32)
    x[::5, 49] = np.inf
    x[1::5, 0] = -np.inf
    _check(crow, col, None, np.ascontiguousarray(x))


@pytest.mark.parametrize("features,mean", [(256, 3), (250, 13), (16, 3)])
def test_spmm_groups_hand_out_rows(features, mean):
    rows = 140000 if features < 64 else 70000
    rng = np.random.default_rng(features)
    lengths = rng.integers(0, 2 * mean + 1, size=rows)
    lengths[:: rows // 7] = 600
    crow, col, rng = _graph(lengths, 1)
    x = rng.standard_normal((rows, features)).astype(np.float32)
    _check(crow, col, None, x)


@pytest.mark.parametrize("long_row", [False, True])
@pytest.mark.parametrize("features", [40, 47, 96, 128, 200])
def test_spmm_rows_known_to_be_even(features, long_row):
    """Above 2^19 edges the op asks for the longest row once per graph."""
    rows = 40000
    lengths = np.full(rows, 14)
    if long_row:
        lengths[777] = 300
    crow, col, rng = _graph(lengths, features)
    assert col.size > 1 << 19
    x = rng.standard_normal((rows, features)).astype(np.float32)
    val = rng.standard_normal(col.size).astype(np.float32)
    d_crow, d_col, d_val, d_x = to_dev(crow, col, val, x)
    assert _native._even_rows(d_crow, d_col, features) is not long_row
    got = torch.ops.autosage.spmm_csr(d_crow, d_col, d_val, d_x)
    ref = oracle.spmm_seq(crow, col, val, x)
    assert bitwise_equal(got, ref), mismatch_report(got, ref)


@pytest.mark.parametrize("rows", [40, 8191, 8192])
@pytest.mark.parametrize("features", [16, 100])
def test_long_rows_start_lower_in_small_graphs(rows, features):
    crow, col, rng = _graph([127, 128, 129, 254, 255, 256, 257, 600] * 4 + [2] * (rows - 32), rows)
    x = rng.standard_normal((rows, features)).astype(np.float32)
    _check(crow, col, None, x)
