"""Labels of batched cuts at the edges of their two forms (a workgroup per
graph, the whole union in memory): graph sizes around 16-bit ids, graphs
without kept edges, many tiny graphs, the padding of a recorded batch. Every
batch is compared, exactly, with the single-graph calls on its graphs."""
import numpy as np
import pytest

from masters_final_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


def _batch(sizes, deg, seed, wmax):
    parts = [synth.random_graph(int(n), min(deg, max(n - 1, 0)), seed + i, wmax=wmax)
             for i, n in enumerate(sizes)]
    goff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    eoff = np.concatenate([[0], np.cumsum([p["dest"].size for p in parts])])
    return parts, {
        "dest": np.concatenate([p["dest"] + goff[i] for i, p in enumerate(parts)]).astype(np.int32),
        "weight": np.concatenate([p["weight"] for p in parts]),
        "indptr": np.concatenate([p["indptr"][:-1] + eoff[i] for i, p in enumerate(parts)]
                                 + [eoff[-1:]]).astype(np.int64), "goff": goff}


def _single(p, rule, max_dist):
    from masters_final_amd._lib import EACError
    from masters_final_amd.graph.singlelink import lifetime_cut
    try:
        lab, info = lifetime_cut(p["dest"], p["weight"], p["indptr"], None, rule=rule,
                                 max_dist=max_dist)
    except (EACError, ValueError):
        return None
    return lab, info


def _check(parts, b, labels, gout, rule, max_dist):
    labels, gout = labels.cpu().numpy(), gout.cpu().numpy()
    for g, p in enumerate(parts):
        want = _single(p, rule, max_dist)
        if want is None:
            assert gout[g, 3] == -1, g
            continue
        lab, info = want
        assert gout[g, 3] == info["kept_edges"] and gout[g, 1] == info["labels_empty"], g
        if lab is not None:
            a, z = b["goff"][g], b["goff"][g + 1]
            assert np.array_equal(labels[a:z], lab.cpu().numpy()), g
            assert gout[g, 0] == info["n_components"], g


@pytest.mark.parametrize("rule,max_dist", [(0, None), (1, None), (1, 30.0)])
@pytest.mark.parametrize("sizes,deg", [
    ([1023, 1024, 1025, 3, 2, 4097], 5), ([65_535, 65_536, 17], 4), ([65_537, 900, 64], 4),
    ([12] * 700, 4), ([16_000, 40_000, 2, 2, 2], 1)])
def test_batches(torch, sizes, deg, rule, max_dist):
    from masters_final_amd.graph.singlelink import LifetimeCutGraph, lifetime_cut_batched
    parts, b = _batch(sizes, deg, 5, 20)
    a = (b["dest"], b["weight"], b["indptr"], b["goff"])
    labels, gout, info = lifetime_cut_batched(*a, rule=rule, max_dist=max_dist)
    if len(sizes) > 100:  # every one of a few
        _check(parts[:40], b, labels, gout[:40], rule, max_dist)
    else:
        _check(parts, b, labels, gout, rule, max_dist)
    want_l, want_g = labels.cpu().numpy(), gout.cpu().numpy()
    assert info["kept_edges"] == want_g[:, 3].clip(0).sum() or (want_g[:, 3] < 0).any()
    assert info["components"] == want_g[:, 0].sum()
    # recorded with room: the padding is one more graph, of isolated vertices
    n, m = int(b["goff"][-1]), b["dest"].size
    cg = LifetimeCutGraph(n + 70_000, m + 9, len(sizes) + 2, torch.int32, rule=rule,
                          max_dist=max_dist)
    for _ in range(3):
        lab, go, inf = cg.run(*a)
        assert np.array_equal(lab.cpu().numpy(), want_l)
        assert np.array_equal(go.cpu().numpy(), want_g)
        assert inf["kept_edges"] == info["kept_edges"]
    cg.close()


@pytest.mark.parametrize("n", [2, 3, 64, 16_000, 16_001, 65_536, 65_537])
def test_single_graph_forms(torch, n):
    """One graph at the limits of the forms, with zero weights, against the
    oracle's rules."""
    from masters_final_amd._lib import EACError
    from masters_final_amd.graph.singlelink import lifetime_cut
    from oracle import oracle as O
    g = synth.random_graph(n, 3, n, wmax=6, n_isolated=n // 50, n_parts=1 + n // 3000)
    rows = np.repeat(np.arange(n), np.diff(g["indptr"]))
    g["weight"][(rows + g["dest"]) % 11 == 0] = 0
    u, v, w, _ = O.csr_edges(g["dest"], g["weight"], g["indptr"][:-1], np.diff(g["indptr"]))
    if not len(u):
        return
    for rule, md in ((1, None), (1, 4.0), (0, None)):
        try:
            if rule == 1:
                want, nc, kept = O.sl_mst_lifetime(u, v, w, n, disconnect_weight=md)
            else:
                nc, want = O.sp_sl_lifetime(u, v, w, n)
                kept = None
        except ValueError:
            with pytest.raises((EACError, ValueError)):
                lifetime_cut(g["dest"], g["weight"], g["indptr"], None, rule=rule, max_dist=md)
            continue
        lab, info = lifetime_cut(g["dest"], g["weight"], g["indptr"], None, rule=rule, max_dist=md)
        if kept is not None:
            assert info["kept_edges"] == kept
        if want.size == 0:
            assert lab is None and info["n_components"] == 1
        else:
            assert info["n_components"] == nc and np.array_equal(lab.cpu().numpy(), want)
