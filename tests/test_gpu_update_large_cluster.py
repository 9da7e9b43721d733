"""Centroid sums of one large cluster, whose rows go through LDS in stages: at
the edges of the stages and with column strides on one bank, against the oracle
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


@pytest.mark.parametrize("d", [1, 5, 11, 33, 36, 37, 43, 52, 61, 64, 66, 100, 129])
def test_stages_of_one_cluster(torch, d):
    from masters_final_amd.cluster.KMeans import update_device
    rng = np.random.default_rng(d)
    dd = min(d, 128)
    rs = min(8192 // dd & ~3, 1024)
    for n in {1, rs - 5, rs - 4, rs - 3, rs, rs + 1, 2 * rs - 4, 2 * rs + 3, 3000}:
        X = (rng.standard_normal((n, d)) * 3).astype(np.float32)
        lab = np.zeros((1, n), np.int32)
        dists = rng.random((1, n)).astype(np.float32)
        got, ne = update_device(X, lab, dists, [1])
        want = O.recompute_centroids(X, lab[0], dists[0], 1, reseed_mode=1)
        assert ne == 0 and np.array_equal(got.cpu().numpy(), want), n


def test_odd_dimensions_cost_about_what_others_do(torch):
    """100,000 points in one cluster, 37-d against 5-d: 4.8 times as long when
    every piece of a row was loaded behind a branch, now twice."""
    import time
    from masters_final_amd.cluster.KMeans import update_device
    n, best = 100_000, {}
    lab = torch.zeros((1, n), dtype=torch.int32, device="cuda")
    dists = torch.rand((1, n), device="cuda")
    for d in (5, 37):
        X = torch.rand((n, d), device="cuda")
        best[d] = float("inf")
        for _ in range(8):
            torch.cuda.synchronize()
            t = time.perf_counter()
            update_device(X, lab, dists, [1])
            torch.cuda.synchronize()
            best[d] = min(best[d], time.perf_counter() - t)
    assert best[37] < 3.3 * best[5]
