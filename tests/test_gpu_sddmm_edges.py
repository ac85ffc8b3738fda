"""The fp32 SDDMM over blocks of 64 edges: every width class of its lanes
(whole and partial 32-feature blocks, multiples of 4 or not, fewer than 4
features), graphs that fill and straddle blocks, 32- and 64-bit offsets.  The
product by rows, which the scheduler may choose."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from autosage_amd import _auto, _native
from gpu_common import bitwise_equal, case_graph, mismatch_report, require_gpu, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


def _graphs():
    yield case_graph(700, 9, seed=5, hubs=3, hub_degree=900, empty=0.1)
    # runs of more than 64 empty rows, then a row across block boundaries
    degrees = np.zeros(1000, dtype=np.int64)
    degrees[[0, 1, 200, 201, 999]] = (1, 63, 130, 1, 62)
    crow = np.concatenate([[0], np.cumsum(degrees)]).astype(np.int64)
    yield crow, np.random.default_rng(1).integers(0, 1000, size=int(crow[-1])).astype(np.int64)
    for nnz in (1, 64, 65):
        crow = np.concatenate([[0], np.full(40, nnz)]).astype(np.int64)
        yield crow, np.random.default_rng(nnz).integers(0, 40, size=nnz).astype(np.int64)


@pytest.mark.parametrize("features", [1, 2, 3, 4, 5, 7, 28, 31, 32, 33, 36, 47, 60, 63, 64, 65, 95, 96, 97, 100, 128,
                                      129, 132, 161, 196, 224, 255, 256, 259, 288, 301])
def test_sddmm_edge_blocks_bitwise(features):
    lib = _native.library()
    for crow, col in _graphs():
        n = crow.size - 1
        rng = np.random.default_rng(features)
        q = rng.standard_normal((n, features)).astype(np.float32)
        k = rng.standard_normal((n, features)).astype(np.float32)
        # an infinity must reach the edges of its own row only, whatever a
        # partial block reads beside its features
        k[0, features - 1] = np.inf
        k[-1, 0] = -np.inf
        ref = oracle.sddmm_ref(crow, col, q, k)
        d_crow, d_col, d_q, d_k = to_dev(crow, col, q, k)
        got = torch.ops.autosage.sddmm_csr(d_crow, d_col, d_q, d_k)
        assert bitwise_equal(got, ref), mismatch_report(got, ref)
        # rows that start 4 bytes off, and the entry that knows no key rows
        off_q, off_k = (torch.empty(t.numel() + 1, device="cuda")[1:].view_as(t).copy_(t) for t in (d_q, d_k))
        out = torch.full((col.size,), float("nan"), device="cuda")
        status = lib.as_sddmm_csr_f32(d_crow.data_ptr(), d_col.data_ptr(), off_q.data_ptr(), off_k.data_ptr(),
                                      out.data_ptr(), n, col.size, features,
                                      torch.cuda.current_stream().cuda_stream)
        assert status == 0
        torch.cuda.synchronize()
        assert bitwise_equal(out, ref), mismatch_report(out, ref)


def test_sddmm_edge_blocks_against_a_larger_key():
    crow, col = case_graph(300, 11, seed=9)
    rng = np.random.default_rng(2)
    col = rng.integers(0, 5000, size=col.size).astype(np.int64)
    q = rng.standard_normal((300, 50)).astype(np.float32)
    k = rng.standard_normal((5000, 50)).astype(np.float32)
    whole_crow = np.concatenate([crow, np.full(4700, crow[-1])]).astype(np.int64)
    ref = oracle.sddmm_ref(whole_crow, col, np.concatenate([q, np.zeros((4700, 50), np.float32)]), k)
    got = _native.sddmm_csr_rect_impl(*to_dev(crow, col, q, k))
    assert bitwise_equal(got, ref), mismatch_report(got, ref)


ROW_LENGTHS = [0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 1022, 1023, 1024, 1025, 2047, 2048, 2049, 4097, 9000, 0]


@pytest.mark.parametrize("features", [32, 64, 96, 128, 160, 192, 224, 256, 48, 288])
@pytest.mark.parametrize("longest", [40, 1024, 9000])
def test_sddmm_by_rows_bitwise(features, longest):
    """Edges in flight and their remainder, rows around the hub and chunk bounds,
    graphs without hub rows; widths and rows that the kernel does not take."""
    rng = np.random.default_rng(features)
    lengths = rng.permutation(np.array([v for v in ROW_LENGTHS if v <= longest] * 3))
    crow = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    n = lengths.size
    col = rng.integers(0, n, size=int(crow[-1])).astype(np.int64)
    q, k = (rng.standard_normal((n, features)).astype(np.float32) for _ in range(2))
    k[0, features - 1], k[-1, 0] = np.inf, np.nan
    ref = oracle.sddmm_ref(crow, col, q, k)
    d_crow, d_col, d_q, d_k = to_dev(crow, col, q, k)
    assert _native.sddmm_rows_supported(d_q, d_k) is (features % 32 == 0 and features <= 256)
    got = torch.ops.autosage.sddmm_csr_rows(d_crow, d_col, d_q, d_k)
    assert np.array_equal(got.cpu().numpy(), ref, equal_nan=True)
    off_k = torch.empty(d_k.numel() + 1, device="cuda")[1:].view_as(d_k).copy_(d_k)
    got = torch.ops.autosage.sddmm_csr_rows(d_crow, d_col, d_q, off_k)
    assert np.array_equal(got.cpu().numpy(), ref, equal_nan=True)


def test_the_scheduler_races_sddmm_by_rows(monkeypatch, tmp_path):
    """Large keys and long rows on average; its gradients, and its replay."""
    monkeypatch.setenv("AUTOSAGE_CACHE_DIR", str(tmp_path))
    crow, col = case_graph(9000, 40, seed=3, hubs=4, hub_degree=5000)
    rng = np.random.default_rng(7)
    q, k = (rng.standard_normal((9000, 64)).astype(np.float32) for _ in range(2))
    d_crow, d_col, d_q, d_k = to_dev(crow, col, q, k)
    assert not _auto._sddmm_rows_eligible(d_crow, d_col, d_q, d_k)
    monkeypatch.setattr(_auto, "_SDDMM_ROWS_MIN_KEY_BYTES", 0)
    assert not _auto._sddmm_rows_eligible(d_crow, d_col[: 31 * 9000], d_q, d_k)
    assert not _auto._sddmm_rows_eligible(d_crow, d_col, d_q[:, :32].contiguous(), d_k[:, :32].contiguous())
    want = oracle.sddmm_ref(crow, col, q, k)
    _, info = _auto.sddmm_csr_auto(d_crow, d_col, d_q, d_k)
    assert "rows" in [c["candidate"] for c in info["full_graph"]["candidates"]]
    leaves = [d_q.requires_grad_(True), d_k.requires_grad_(True)]
    grad = torch.randn(col.size, device="cuda")
    results = []
    for candidate in ("rows", info["candidate"]):
        assert _auto._cached_native_available("sddmm_csr", "autosage", candidate)
        out = _auto._run_sddmm_choice("autosage", candidate, d_crow, d_col, *leaves)
        assert bitwise_equal(out, want)
        results.append(torch.autograd.grad(out, leaves, grad))
    assert all(torch.equal(a, b) for a, b in zip(*results))
