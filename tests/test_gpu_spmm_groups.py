"""The fp32 whole-graph SpMM in lane groups and workgroups on long rows, bit
for bit against the sequential product: widths around the lane and slice
bounds, rows around the batch, tile and long-row bounds, rows handed out
within a wave, one wave per row on graphs known to be even."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import autosage_amd
import oracle
from autosage_amd import _autograd, _native, shard
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
    """Above 2^19 edges the op asks for the longest row once per graph, and knows
    it from the next call on that finds the answer."""
    rows = 40000
    lengths = np.full(rows, 14)
    if long_row:
        lengths[777] = 300
    crow, col, rng = _graph(lengths, features)
    assert col.size > 1 << 19
    x = rng.standard_normal((rows, features)).astype(np.float32)
    val = rng.standard_normal(col.size).astype(np.float32)
    d_crow, d_col, d_val, d_x = to_dev(crow, col, val, x)
    ref = oracle.spmm_seq(crow, col, val, x)
    for known in (False, not long_row, not long_row):
        torch.cuda.synchronize()
        assert _native._even_rows(d_crow, d_col, features) is known
        got = torch.ops.autosage.spmm_csr(d_crow, d_col, d_val, d_x)
        assert bitwise_equal(got, ref), mismatch_report(got, ref)


def _even_graph(features):
    rows = 40000
    crow, col, rng = _graph(np.full(rows, 14), features)
    x = rng.standard_normal((rows, features)).astype(np.float32)
    return to_dev(crow, col, x), oracle.spmm_seq(crow, col, None, x)


def test_no_call_waits_for_the_longest_row():
    """A new graph, its transpose in the backward and int32 indices, in the range
    where the longest row matters: nothing waits for the device."""
    (crow, col, x), ref = _even_graph(64)
    autosage_amd.spmm_csr(*(t.clone() for t in (crow, col)), None, x)  # loads what the first call loads
    x.requires_grad_(True)
    crow_t, col_t, _ = _autograd.csr_transpose(crow, col)
    mode = torch.cuda.get_sync_debug_mode()
    torch.cuda.set_sync_debug_mode("error")
    try:
        out = [autosage_amd.spmm_csr(crow, col, None, x)]
        (grad,) = torch.autograd.grad(out[0], (x,), x.detach())
        for _ in range(2):
            out.append(autosage_amd.spmm_csr(crow.int(), col.int(), None, x))
    finally:
        torch.cuda.set_sync_debug_mode(mode)
    assert all(bitwise_equal(o, ref) for o in out)
    assert torch.equal(grad, torch.ops.autosage.spmm_csr(crow_t, col_t, None, x.detach()))


def test_nothing_is_asked_about_copies_and_widths_without_a_choice(monkeypatch):
    (crow, col, x), _ = _even_graph(64)
    entries = len(_native._LONGEST_ROW_MEMO)
    autosage_amd.spmm_csr(crow.int(), col.int(), None, x)
    shard.spmm_csr_shard(crow.int(), col.int(), None, x, exact=True)
    assert not _native._even_rows(crow, col, 65) and not _native._even_rows(crow, col, 32)
    monkeypatch.setenv("AUTOSAGE_VEC4", "0")
    assert not _native._even_rows(crow, col, 64)
    assert len(_native._LONGEST_ROW_MEMO) == entries


@pytest.mark.parametrize("exact_shard", [False, True])
def test_graphs_made_in_inference_mode(exact_shard):
    """Tensors without a version counter."""
    with torch.inference_mode():
        (crow, col, x), ref = _even_graph(64)
        call = ((lambda: _native.spmm_csr_rect_impl(crow, col, None, x, exact=True)) if exact_shard
                else (lambda: autosage_amd.spmm_csr(crow, col, None, x)))
        assert crow.is_inference()
        for _ in range(2):
            assert bitwise_equal(call(), ref)
    assert bitwise_equal(call(), ref)


def test_the_longest_row_under_capture():
    (crow, col, x), ref = _even_graph(64)
    torch.ops.autosage.spmm_csr(crow.clone(), col, None, x)  # loads the kernels
    y = torch.zeros_like(x)
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    for graph in graphs:  # nobody asked; then the answer is there
        with torch.cuda.graph(graph):
            y.copy_(torch.ops.autosage.spmm_csr(crow, col, None, x))
        for _ in range(2):
            y.zero_()
            graph.replay()
            assert bitwise_equal(y, ref)
        torch.ops.autosage.spmm_csr(crow, col, None, x)
        torch.cuda.synchronize()
        assert _native._even_rows(crow, col, 64)


@pytest.mark.parametrize("rows", [40, 8191, 8192])
@pytest.mark.parametrize("features", [16, 100])
def test_long_rows_start_lower_in_small_graphs(rows, features):
    crow, col, rng = _graph([127, 128, 129, 254, 255, 256, 257, 600] * 4 + [2] * (rows - 32), rows)
    x = rng.standard_normal((rows, features)).astype(np.float32)
    _check(crow, col, None, x)
