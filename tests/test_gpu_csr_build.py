"""The native CSR build and transpose against the torch composition, integer
for integer: sizes on both sides of the sort's bounds, empty rows, ids at the
ends of the key bits, hubs, views; ids outside the rows; what keeps the torch
composition."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from autosage_amd import _autograd, _native
from autosage_amd.utils.csr import csr_with_edge_order, edge_index_to_csr
from gpu_common import case_graph, require_gpu, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.mark.parametrize("nodes,edges", [(1, 1), (1, 700), (2, 65), (255, 4000), (256, 65535), (257, 65536), (4000, 65537),
                                         (65535, 70000), (65536, 70000), (65537, 300000), (300, 4000001)])
def test_native_csr_build_equals_the_torch_steps(nodes, edges):
    rng = np.random.default_rng(nodes + edges)
    ids = rng.integers(0, nodes, size=(2, edges))
    ids[:, 0] = nodes - 1
    ids[1, edges // 3: edges // 2] = nodes // 2  # a hub
    host = torch.from_numpy(ids)
    dev = host.cuda()
    assert _native.csr_build_supported(dev[1], dev[0], nodes)
    for rows_by in ("dst", "src"):
        want = csr_with_edge_order(host, nodes, rows_by=rows_by)  # the CPU's torch steps
        got = csr_with_edge_order(dev, nodes, rows_by=rows_by)
        assert all(torch.equal(g.cpu(), w) for g, w in zip(got, want))
        crow, col = edge_index_to_csr(dev.t().contiguous().t(), nodes, rows_by=rows_by)  # strided ids
        assert torch.equal(crow.cpu(), want[0]) and torch.equal(col.cpu(), want[1])
        crow, col = edge_index_to_csr(dev.to(torch.int32), nodes, rows_by=rows_by)
        assert torch.equal(crow.cpu(), want[0]) and torch.equal(col.cpu(), want[1])
    crow, col = want[0], want[1]
    got_t = _autograd._build_transpose(crow.cuda(), col.cuda())
    assert all(torch.equal(g.cpu(), w) for g, w in zip(got_t, _autograd._build_transpose(crow, col)))


def test_native_transpose_of_graphs_with_empty_rows():
    for seed, empty in ((1, 0.0), (2, 0.9)):
        crow, col = case_graph(5000, 12, seed=seed, hubs=3, hub_degree=3000, empty=empty)
        host = _autograd._build_transpose(torch.from_numpy(crow), torch.from_numpy(col))
        dev = _autograd._build_transpose(*to_dev(crow, col))
        assert all(torch.equal(d.cpu(), h) for d, h in zip(dev, host))


def test_ids_outside_the_rows_end_behind_the_last_row():
    rows = torch.tensor([3, -1, 0, 4, 2, 1 << 40, 0], device="cuda")
    cols = torch.arange(7, device="cuda")
    crow, col, perm = _native.csr_from_edges(rows, cols, 4)
    assert crow.tolist() == [0, 2, 2, 3, 4]
    assert col.tolist() == [2, 6, 4, 0, 1, 3, 5] and perm.tolist() == col.tolist()


def test_what_keeps_the_torch_composition():
    ids = torch.zeros(4, dtype=torch.long, device="cuda")
    assert _native.csr_build_supported(ids, ids, 3)
    assert not _native.csr_build_supported(ids[:0], ids[:0], 3)  # no edges
    assert not _native.csr_build_supported(ids, ids, 0)
    assert not _native.csr_build_supported(ids[::2], ids[::2], 3)
    seen = []
    torch.func.vmap(lambda t: seen.append(_native.csr_build_supported(t, t, 3)) or t)(ids.view(1, 4))
    assert seen == [False]
    empty = torch.zeros((2, 0), dtype=torch.long, device="cuda")
    crow, col = edge_index_to_csr(empty, 3)
    assert crow.tolist() == [0, 0, 0, 0] and col.numel() == 0
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = _native.csr_build_supported(ids, ids, 3)
    assert not captured
