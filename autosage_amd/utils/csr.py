"""edge_index -> CSR with destination rows (``autosage/utils/csr.py:6-26``).

Rows are ``edge_index[1]`` (destinations) by default.  Edges are ordered by a
stable sort of the row ids, so within a row the columns keep their edge_index
order; ``crow`` is the cumulative count of edges per row.  Integer-only and
identical on CPU and GPU.  On the CPU the steps (stable argsort,
``index_add_`` of ones at row + 1, ``cumsum``) are the reference's, because the
output must be bit-identical to it; on the GPU one native sort gives the same
integers (``_native.csr_from_edges``), with those steps as the fallback under
tracing and stream capture.
"""

from __future__ import annotations

import torch


def _row_and_column_ids(edge_index: torch.Tensor, rows_by: str) -> tuple[torch.Tensor, torch.Tensor]:
    if edge_index.ndim != 2 or edge_index.size(0) != 2:
        raise ValueError("edge_index must have shape [2, E]")
    if rows_by not in ("dst", "src"):
        raise ValueError("rows_by must be 'dst' or 'src'")
    src = edge_index[0].to(dtype=torch.long)
    dst = edge_index[1].to(dtype=torch.long)
    return (dst, src) if rows_by == "dst" else (src, dst)


def _native_csr(rows: torch.Tensor, cols: torch.Tensor, num_nodes: int, want_order: bool):
    """(crow, col, order) from the native build, or Nones where it does not
    apply (see ``_native.csr_build_supported``)."""
    if not rows.is_cuda or torch.compiler.is_compiling():
        return None, None, None
    from .. import _native
    from ..ops import load_native

    load_native()
    rows_c, cols_c = rows.contiguous(), cols.contiguous()
    if not isinstance(num_nodes, int) or not _native.csr_build_supported(rows_c, cols_c, num_nodes):
        return None, None, None
    built = _native.csr_from_edges_checked(rows_c, cols_c, num_nodes, want_order)
    if built is None:
        # an id outside [0, num_nodes): refused as on the CPU, but for -1, which
        # the torch steps count ahead of the first row
        if bool(((rows < -1) | (rows >= num_nodes)).any()):
            raise IndexError("edge_index holds a node id outside [0, num_nodes)")
        return None, None, None
    return built


def csr_with_edge_order(
    edge_index: torch.Tensor,
    num_nodes: int,
    *,
    rows_by: str = "dst",
) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(crow, col, order): the CSR of ``edge_index_to_csr`` and the edge
    permutation that produced it — CSR position k holds edge ``order[k]`` of
    ``edge_index`` — so per-edge data (weights) follows with one
    ``index_select``."""
    rows, cols = _row_and_column_ids(edge_index, rows_by)
    crow, col, order = _native_csr(rows, cols, num_nodes, True)
    if crow is not None:
        return crow, col, order
    order = rows.argsort(stable=True)
    counts = torch.zeros(num_nodes + 1, dtype=torch.long, device=rows.device)
    # integer counts: the order of the additions does not matter
    counts.index_add_(0, rows + 1, torch.ones_like(rows))
    return counts.cumsum(0).contiguous(), cols.index_select(0, order).contiguous(), order


def edge_index_to_csr(
    edge_index: torch.Tensor,
    num_nodes: int,
    *,
    rows_by: str = "dst",
) -> tuple[torch.Tensor, torch.Tensor]:
    rows, cols = _row_and_column_ids(edge_index, rows_by)
    crow, col, _ = _native_csr(rows, cols, num_nodes, False)
    if crow is None:
        crow, col, _ = csr_with_edge_order(edge_index, num_nodes, rows_by=rows_by)
    return crow, col


__all__ = ["csr_with_edge_order", "edge_index_to_csr"]
