"""Cuts of paths whose vertices are in order (sorted one-dimensional data, time
series): the first hooking makes one chain of every kept stretch. Against the
cut's definition: the heaviest edges go, the stretches are numbered in order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


def _path(torch, w, order=None):
    """CSR of a path with these edge weights, its vertices renamed by order."""
    n = len(w) + 1
    at = np.arange(n) if order is None else order
    u, v = at[:-1], at[1:]
    r, c = np.concatenate([u, v]), np.concatenate([v, u])
    o = np.lexsort((c, r))
    ww = np.concatenate([w, w])[o]
    ip = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))])
    return [torch.from_numpy(np.ascontiguousarray(x)).cuda()
            for x in (c[o].astype(np.int32), ww.astype(np.int32), ip.astype(np.int64))]


@pytest.mark.parametrize("n", [2, 17, 18, 34, 300, 5000, 49_152])
@pytest.mark.parametrize("kind", ["up", "down", "mixed"])
def test_cut_of_a_path_in_order(torch, n, kind):
    from masters_final_amd.graph.singlelink import lifetime_cut, lifetime_cut_batched
    rng = np.random.default_rng(n)
    w = {"up": np.arange(1, n), "down": np.arange(n - 1, 0, -1),
         "mixed": rng.permutation(n - 1) + 1}[kind]
    dest, ww, ip = _path(torch, w)
    for c in {2, min(5, n), max(2, n // 3)}:
        cut = np.zeros(n, np.int64)
        cut[1:][np.argsort(w)[n - c:]] = 1  # the c - 1 heaviest edges
        want = np.cumsum(cut).astype(np.int32)
        if n > 2:
            lab, info = lifetime_cut(dest, ww, ip, rule=0, max_dist=1e9, n_clusters=c)
            assert info["n_components"] == c and np.array_equal(lab.cpu().numpy(), want)
    if n == 5000:  # several of them, one workgroup each
        m = dest.numel()
        d3 = torch.cat([dest + i * n for i in range(3)])
        ip3 = torch.cat([ip[:-1] + i * m for i in range(3)] + [torch.tensor([3 * m]).cuda()])
        lab, gout, _ = lifetime_cut_batched(d3, ww.repeat(3), ip3, np.arange(4) * n,
                                            max_dist=1e9, n_clusters=c)
        assert np.array_equal(lab.cpu().numpy(), np.tile(want, 3))


def test_order_of_the_vertices_costs_little(torch):
    """The same path with its vertices in order and shuffled: walks to the root
    took 19 times as long in order, in steps about as long."""
    import time
    from masters_final_amd.graph.singlelink import lifetime_cut
    n, best = 48_000, {}
    rng = np.random.default_rng(1)
    w = rng.permutation(n - 1) + 1
    for name, order in (("in order", None), ("shuffled", rng.permutation(n))):
        g = _path(torch, w, order)
        best[name] = float("inf")
        for _ in range(8):
            torch.cuda.synchronize()
            t = time.perf_counter()
            lifetime_cut(*g, rule=0, max_dist=1e9, n_clusters=5)
            torch.cuda.synchronize()
            best[name] = min(best[name], time.perf_counter() - t)
    assert best["in order"] < 5 * best["shuffled"]
