"""The exact attention's three launches against the three operators: feature
widths at the edges of their kernels' ranges, a scale that rounds, rows of
every kind of the softmax, whose scores the call overwrites in place."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import autosage_amd
from gpu_common import require_gpu, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    require_gpu()


@pytest.mark.parametrize("fqk, fv", [(1, 1), (3, 3), (4, 4), (33, 5), (100, 47), (520, 260)])
@pytest.mark.parametrize("scale", [1.0, 0.1767767])
def test_attention_equals_its_stages(fqk, fv, scale):
    rng = np.random.default_rng(fqk)
    lengths = rng.permutation(np.array([0, 1, 16, 64, 65, 255, 256, 513, 4096, 4097, 0, 9001] + [7] * 300))
    n = lengths.size
    crow = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    col = rng.integers(0, n, size=int(crow[-1])).astype(np.int64)
    q, k, v = (rng.standard_normal((n, f)).astype(np.float32) for f in (fqk, fqk, fv))
    d = to_dev(crow, col, q, k, v)
    got = torch.ops.autosage.csr_attention(*d, scale)
    scores = torch.ops.autosage.sddmm_csr(*d[:4]) * np.float32(scale).item()
    probs = torch.ops.autosage.csr_row_softmax(d[0], scores)
    assert torch.equal(got, torch.ops.autosage.spmm_csr(d[0], d[1], probs, d[4]))


@pytest.mark.parametrize("which", ["qkv", "q", "k", "v"])
def test_backward_with_the_forwards_probabilities(which):
    """The gradients of the op that recomputes them, bit for bit, also where a
    graph is recorded through the backward; the probabilities have no gradient."""
    rng = np.random.default_rng(5)
    lengths = rng.permutation(np.array([0, 1, 65, 4097, 0] + [9] * 200))
    n = lengths.size
    crow = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    col = rng.integers(0, n, size=int(crow[-1])).astype(np.int64)
    d_crow, d_col = to_dev(crow, col)
    leaves = [t.requires_grad_(name in which) for name, t in
              zip("qkv", to_dev(*(rng.standard_normal((n, f)).astype(np.float32) for f in (20, 20, 33))))]
    wanted = [t for t in leaves if t.requires_grad]
    ops = torch.ops.autosage
    ref = ops.csr_attention(d_crow, d_col, *leaves, 0.3)
    out, probs = ops.csr_attention_probs(d_crow, d_col, *leaves, 0.3)
    assert torch.equal(out, ref) and not probs.requires_grad
    g = torch.randn_like(ref)
    want = torch.autograd.grad(ref, wanted, g)
    again = torch.autograd.grad(out, wanted, g, create_graph=True)
    assert all(torch.equal(a, w) for a, w in zip(again, want))
    got = torch.autograd.grad(out, wanted, g)
    assert all(torch.equal(a, w) for a, w in zip(got, want))


@pytest.mark.parametrize("fqk", [0, 8])
def test_values_of_no_width_have_zero_gradients(fqk):
    """Scores and probabilities exist without value features; the gradients of
    query and key are 0 whatever the memory held before."""
    rng = np.random.default_rng(3)
    lengths = np.array([5, 0, 300, 40] * 50)
    n = lengths.size
    crow = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    col = rng.integers(0, n, size=int(crow[-1])).astype(np.int64)
    d_crow, d_col, q, k, v = to_dev(crow, col, *(rng.standard_normal((n, f)).astype(np.float32) for f in (fqk, fqk, 0)))
    leaves = [q.requires_grad_(True), k.requires_grad_(True)]
    for call in (lambda: torch.ops.autosage.csr_attention_probs(d_crow, d_col, q, k, v, 0.5),
                 lambda: autosage_amd.csr_attention_forward(d_crow, d_col, q, k, v, scale=0.5),
                 lambda: (torch.ops.autosage.csr_attention(d_crow, d_col, q, k, v, 0.5),)):
        for _ in range(4):  # freed blocks of this size hold NaN
            torch.full((col.size,), float("nan"), device="cuda")
        out = call()[0]
        assert out.shape == (n, 0)
        for grad in torch.autograd.grad(out, leaves, torch.empty_like(out)):
            assert grad.shape == (n, fqk) and not grad.any()
    _, probs = torch.ops.autosage.csr_attention_probs(d_crow, d_col, q, k, v, 0.5)
    scores = torch.ops.autosage.sddmm_csr(d_crow, d_col, q, k) * 0.5
    assert torch.equal(probs, torch.ops.autosage.csr_row_softmax(d_crow, scores))


def test_attention_without_edges_is_zero():
    crow, col = torch.zeros(6, dtype=torch.long, device="cuda"), torch.empty(0, dtype=torch.long, device="cuda")
    q, v = torch.ones(5, 8, device="cuda"), torch.ones(5, 12, device="cuda")
    assert not torch.ops.autosage.csr_attention(crow, col, q, q, v, 1.0).any()
