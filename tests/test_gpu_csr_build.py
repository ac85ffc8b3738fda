"""The native CSR build and transpose against the torch composition, integer
for integer: sizes on both sides of the sort's bounds, empty rows, ids at the
ends of the key bits, hubs, views; ids outside the rows; what keeps the torch
composition."""

from __future__ import annotations

import numpy as np
import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx

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


@pytest.mark.parametrize("edges", [1, 700, 300000])
@pytest.mark.parametrize("bad", [None, 500, -2, 1 << 40, -1])
def test_ids_outside_the_nodes_are_refused_as_on_the_cpu(edges, bad):
    nodes = 500
    ids = torch.from_numpy(np.random.default_rng(edges).integers(0, nodes, size=(2, edges)))
    ids[:, edges // 2] = nodes - 1
    for rows_by, end in (("dst", 1), ("src", 0)):
        host = ids.clone()
        if bad is not None:
            host[end, edges * 2 // 3] = bad
        for build in (edge_index_to_csr, csr_with_edge_order):
            if bad is None or bad == -1:  # -1 is counted ahead of the first row
                want = build(host, nodes, rows_by=rows_by)
                got = build(host.cuda(), nodes, rows_by=rows_by)
                assert all(torch.equal(g.cpu(), w) for g, w in zip(got, want))
            else:
                for where in (host, host.cuda()):
                    with pytest.raises(IndexError):
                        build(where, nodes, rows_by=rows_by)


@pytest.mark.parametrize("what", ["column n", "column -1", "far column", "edges past the last row", "descending"])
def test_malformed_graphs_have_no_transpose(what):
    crow, col = case_graph(3000, 20, seed=4)
    if "column" in what:
        col[col.size // 2] = {"column n": 3000, "column -1": -1, "far column": 1 << 33}[what]
    elif what == "descending":
        crow[1500] = crow[-1]
    else:
        crow[-1] -= 1
    d = to_dev(crow, col)
    assert _native.csr_build_supported(*d, 3000)
    with pytest.raises(RuntimeError, match="malformed CSR"):
        _autograd._build_transpose(*d)
    # the next call is not affected
    crow, col = case_graph(3000, 20, seed=4)
    host = _autograd._build_transpose(torch.from_numpy(crow), torch.from_numpy(col))
    assert all(torch.equal(d.cpu(), h) for d, h in zip(_autograd._build_transpose(*to_dev(crow, col)), host))


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
    traced = make_fx(lambda e: edge_index_to_csr(e, 3))(torch.tensor([[0, 1, 2], [2, 2, 0]], device="cuda"))
    other = torch.tensor([[1, 0, 2], [0, 1, 0]], device="cuda")
    assert all(torch.equal(t, e) for t, e in zip(traced(other), edge_index_to_csr(other, 3)))
    compiled = torch.compile(lambda e: edge_index_to_csr(e, 3), backend="eager", fullgraph=True)
    assert all(torch.equal(t, e) for t, e in zip(compiled(other), edge_index_to_csr(other, 3)))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = _native.csr_build_supported(ids, ids, 3)
    assert not captured
