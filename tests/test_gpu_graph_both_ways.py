"""Forests of small graphs passed as not symmetric, on both sides of the entries
one workgroup takes then, against the oracle's canonical Kruskal forest."""
import numpy as np
import pytest
from test_gpu_graph import _check_forest

from masters_final_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [0, 2])  # entries: 180,224 and two more
@pytest.mark.parametrize("wmax", [1, 50])
def test_entries_around_the_limit(extra, wmax):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from masters_final_amd.graph.mst import boruvka_mst
    n, half = 3000, (176 * 1024 + extra) // 2
    rng = np.random.default_rng(wmax)
    u, v = rng.integers(0, n, 3 * half), rng.integers(0, n, 3 * half)
    pick = np.unique((np.minimum(u, v).astype(np.int64) * n + np.maximum(u, v))[u != v])
    pick = rng.permutation(pick)[:half]
    ip, dest, w = synth.csr_from_undirected(n, (pick // n).astype(np.int32),
                                            (pick % n).astype(np.int32),
                                            rng.integers(1, wmax + 1, half).astype(np.int32))
    g = {"n": n, "dest": dest, "weight": w, "indptr": ip}
    assert g["dest"].size == 176 * 1024 + extra
    a = boruvka_mst(g["dest"], g["weight"], g["indptr"], None, symmetric=False,
                    want_weights=True, want_labels=True)
    _check_forest(g, a)
