"""Forests of graphs that fit one workgroup, at the edges of that form, against
the oracle's canonical Kruskal forest and components (all values are integers:
exact)."""
import numpy as np
import pytest
from test_gpu_graph import _check_forest

from masters_final_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.mark.parametrize("n,deg,wmax", [
    (1, 1, 3), (2, 1, 3), (3, 1, 3), (64, 4, 2), (1023, 3, 5), (1024, 9, 1000), (1025, 6, 5),
    (6000, 14, 200), (15_999, 3, 1000), (16_000, 8, 60_000), (16_000, 40, 100),
    (16_001, 8, 60_000)])
def test_small_forests(torch, n, deg, wmax):
    from masters_final_amd.graph.mst import boruvka_mst
    g = synth.random_graph(n, deg, n + deg, wmax=wmax, n_isolated=n // 9, n_parts=1 + n // 500)
    dest, w = torch.from_numpy(g["dest"]).cuda(), torch.from_numpy(g["weight"]).cuda()
    fe = torch.from_numpy(g["indptr"]).cuda()
    a = boruvka_mst(dest, w, fe, None, want_weights=True, want_labels=True)
    _check_forest(g, a)
    b = boruvka_mst(dest, w, fe[:-1].contiguous(), (fe[1:] - fe[:-1]).to(torch.int32),
                    want_weights=False, want_labels=False)
    assert b["n_mst"] == a["n_mst"] and torch.equal(b["ids"][:b["n_mst"]], a["ids"][:a["n_mst"]])
    assert a["rounds"] == b["rounds"]


@pytest.mark.parametrize("direction", [-1, 1])
def test_small_long_pick_chain(torch, direction):
    """A path of ascending weights: one pick chain through every vertex."""
    from masters_final_amd.graph.mst import boruvka_mst
    n = 16_000
    w1 = np.arange(1, n, dtype=np.int32)[::direction]
    u = np.arange(n - 1, dtype=np.int32)
    rows, cols = np.concatenate([u, u + 1]), np.concatenate([u + 1, u])
    w = np.concatenate([w1, w1])
    o = np.lexsort((cols, rows))
    g = {"n": n, "dest": cols[o], "weight": w[o],
         "indptr": np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])}
    r = boruvka_mst(g["dest"], g["weight"], g["indptr"], None, want_weights=True,
                    want_labels=True)
    _check_forest(g, r)
    assert r["rounds"] == 2


@pytest.mark.parametrize("length", [3, 4, 16, 999])
def test_small_pick_cycle_is_reported(torch, length):
    from masters_final_amd._lib import EACError
    from masters_final_amd.graph.mst import boruvka_mst
    dest = np.roll(np.arange(length), -1).astype(np.int32)
    # every row lists only the next vertex; its own entry is its lightest
    with pytest.raises(EACError, match="not symmetric"):
        boruvka_mst(dest, np.ones(length, np.int32), np.arange(length + 1), None,
                    symmetric=True, want_labels=True)
