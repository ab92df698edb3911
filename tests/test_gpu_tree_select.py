"""dtree_tree_build where its top-k bound and its heap's registers can go wrong:
the largest logits inside one thread's 32, equal ones at and past the 256
candidates the bound may pass, k = 1 and 127, vocabularies with fewer threads
than k, negative-only and -inf logits in the list, and heaps past 64 entries
whose scores tie exactly (ranks decide). Ids, nodes and bitsets are exact."""
import numpy as np
import pytest
import torch

from oracle import tree as otree

from dtree_hip import _native as N
from dtree_hip.engine import ancestor_bitsets
from test_gpu_tree import _run

pytestmark = pytest.mark.gpu


def _rows(kind, D, V, seed):
    g = np.random.default_rng(seed)
    x = g.standard_normal((D, V)).astype(np.float32)
    if kind == "cluster":  # the top 32 and a few equal values next to each other
        x[:, 64:96] += 20.0
        x[:, 70:74] = 30.0
    elif kind.startswith("equal"):  # n equal maxima
        n = int(kind[5:])
        x[:, g.permutation(V)[:n]] = 7.0
    elif kind == "same":
        x[:] = 0.25
    elif kind == "negative":
        x = -np.abs(x) - 1e-3
    elif kind == "fewfinite":
        x[:, 3:] = -np.inf
    return x


@pytest.mark.parametrize("kind,D,V,k,budget", [
    ("cluster", 3, 20000, 24, 24), ("cluster", 2, 8192, 127, 100), ("equal255", 2, 30000, 24, 24),
    ("equal256", 2, 8192, 30, 30), ("equal257", 2, 8192, 30, 30), ("same", 18, 9000, 127, 127),
    ("same", 3, 300, 127, 127), ("negative", 4, 8196, 1, 4), ("negative", 15, 33000, 127, 127),
    ("fewfinite", 2, 64, 4, 6), ("normal", 18, 16384, 65, 65)])
def test_select_and_heap_edges(gpu_device, kind, D, V, k, budget):
    print(f"tree select kind={kind} D={D} V={V} k={k} budget={budget}", flush=True)
    x = _rows(kind, D, V, D + V + k)
    ids, lps, out, rec = _run(torch.from_numpy(x).to(gpu_device), k, budget, 5, 70)
    assert np.array_equal(ids, otree._topk_sorted(x, k)[0])
    node_ids, depths, parents, _, _ = otree.heap_tree(ids.astype(np.int64), lps, budget)
    n, M = len(node_ids), N.MAX_NODES
    assert int(out[0]) == n and out[1:1 + n].tolist() == node_ids and out[1 + M:1 + M + n].tolist() == depths
    assert rec["parents"][:n + 1].tolist() == parents
    assert np.array_equal(rec["ancestors"][:n + 1], ancestor_bitsets(parents))
    assert not rec["ancestors"][n + 1:].any() and not out[1 + n:M].any()
