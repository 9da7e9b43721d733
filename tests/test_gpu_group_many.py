"""Grouping with thousands of clusters a partition (radix passes instead of the
counting sort, whose wavefronts would walk chunks as long as four times the
clusters), on both sides of the rule, against the oracle
(MyML/MyML/cluster/KMeans.py:709-754)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.mark.parametrize("n,ks", [
    (2200, [801]), (2201, [801]),             # the last radix size, the first counted one
    (1500, [1, 3000, 2, 900]),                # uneven, empty clusters
    (20_000, [5000, 9000]),
    (1, [4000]),
])
def test_update_on_both_sides_of_the_rule(torch, n, ks):
    from masters_final_amd.cluster.KMeans import update_device
    rng = np.random.default_rng(n)
    X = (rng.standard_normal((n, 3)) * 3).astype(np.float32)
    lab = np.stack([rng.integers(0, min(k, n), n) for k in ks]).astype(np.int32)
    dists = rng.random((len(ks), n)).astype(np.float32)
    empty = [int(np.sum(np.bincount(lab[p], minlength=k) == 0)) for p, k in enumerate(ks)]
    if max(empty) > n:  # more empty clusters than points to reseed them from
        from masters_final_amd._lib import EACError
        with pytest.raises(EACError, match="more empty clusters"):
            update_device(X, lab, dists, ks)
        return
    got, ne = update_device(X, lab, dists, ks)
    got = got.cpu().numpy()
    at = 0
    for p, k in enumerate(ks):
        want = O.recompute_centroids(X, lab[p], dists[p], k, reseed_mode=1)
        assert np.array_equal(got[at:at + k], want), p
        at += k
    assert ne == sum(empty)


@pytest.mark.parametrize("n,P,k", [(3000, 2, 2900), (40_000, 1, 30_000)])
def test_plan_of_many_clusters(torch, n, P, k):
    from masters_final_amd._lib import EACError
    from masters_final_amd.EAC.sparse import coassoc_device
    rng = np.random.default_rng(n)
    lab = rng.integers(-1, k, (P, n)).astype(np.int32)
    ip, ind, dat, _ = coassoc_device(lab, [k] * P)
    wi, wc, wd = O.coassoc_condensed(lab, [k] * P)
    assert np.array_equal(ip.cpu().numpy(), wi)
    assert np.array_equal(ind.cpu().numpy(), wc) and np.array_equal(dat.cpu().numpy(), wd)
    lab[-1, 5] = k
    with pytest.raises(EACError, match="label >= k"):
        coassoc_device(lab, [k] * P)


def test_many_clusters_cost_about_what_few_do(torch):
    """An update of 1,000,000 points with 50,000 clusters against 500: the
    counting sort alone took 20 times as long, the radix passes about as long."""
    import time
    from masters_final_amd.cluster.KMeans import update_device
    n, best = 1_000_000, {}
    X = torch.rand((n, 2), device="cuda")
    dists = torch.rand((1, n), device="cuda")
    for k in (500, 50_000):
        lab = (torch.arange(n, device="cuda", dtype=torch.int32) % k)[None].contiguous()
        best[k] = float("inf")
        for _ in range(8):
            torch.cuda.synchronize()
            t = time.perf_counter()
            update_device(X, lab, dists, [k])
            torch.cuda.synchronize()
            best[k] = min(best[k], time.perf_counter() - t)
    assert best[50_000] < 6 * best[500]
