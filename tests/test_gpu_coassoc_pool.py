"""The one-visit build's pool when it holds every pair: a place for each and no
more, and the matrix of the two-visit build from it, at the edges of windows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.mark.parametrize("n", [1, 2, 4096, 10_000, 23_170])
@pytest.mark.parametrize("full", [0, 1])
def test_pool_for_every_pair_takes_four_bytes_each(torch, n, full):
    """At 10,000 points the chunks of the resident workgroups, which such a
    pool does not need, came to 1.15 GB beside 0.2 GB of pairs."""
    from masters_final_amd import _lib as L
    lib = L.load_library()
    pairs = n * (n - 1) // (1 if full else 2)
    windows = -(-n // 16384)
    for entries in (pairs, pairs + 12345):
        nb = lib.eac_coassoc_stage_bytes(n, full, 100, entries)
        assert 4 * pairs <= nb <= 4 * pairs + 8 * windows * n + 512
    assert pairs == 0 or lib.eac_coassoc_stage_bytes(n, full, 100, pairs - 1) > 4 * (pairs - 1)


@pytest.mark.parametrize("n,P,k,full,window", [
    (4100, 9, 1, False, 0), (4100, 3, 1, True, 0),       # every pair an entry
    (4100, 9, 40, False, 512), (4100, 9, 40, True, 512),  # rows over several windows
    (4103, 300, 700, True, 512),                          # 16-bit counters
    (20_000, 3, 30, False, 0),                            # two windows
])
def test_matrix_from_a_pool_for_every_pair(torch, n, P, k, full, window):
    from masters_final_amd.EAC.sparse import coassoc_device
    from masters_final_amd.tune import get_knobs, set_knobs
    rng = np.random.default_rng(n + k)
    labels = rng.integers(0, k, (P, n)).astype(np.int32)
    labels[0, ::11] = -1  # samples not listed
    saved = get_knobs()
    try:
        if window:
            set_knobs(co_window=window)
        info = {}
        a = coassoc_device(labels, [k] * P, full_rows=full, info=info)
        b = coassoc_device(labels, [k] * P, full_rows=full, one_pass=False)
    finally:
        set_knobs(**saved)
    assert info["path"] == ("one-pass" if n < 16_384 or not full else "two-pass")
    assert a[3] == b[3]
    for x, y in zip(a[:3], b[:3]):
        assert torch.equal(x, y)


@pytest.mark.parametrize("seed", [1, 2])
def test_recorded_build_with_a_pool_for_every_pair(torch, seed):
    """EnsembleCoassocGraph's default capacity, replayed, against the eager run."""
    from masters_final_amd.EAC.eac import EnsembleCoassocGraph
    from masters_final_amd.EAC.sparse import coassoc_device
    from masters_final_amd.utils.partition import generate_ensemble_batched
    g = torch.Generator(device="cuda").manual_seed(seed)
    X = torch.randn((3000, 2), generator=g, device="cuda")
    ks = [20, 30, 7]
    init = torch.cat([X[torch.randperm(3000, generator=g, device="cuda")[:k]] for k in ks])
    rec = EnsembleCoassocGraph(X, ks)
    for it in range(3):
        got = rec.run(init + 0.01 * it)
        labels, _ = generate_ensemble_batched(X, ks, iters=3, init=init + 0.01 * it)
        want = coassoc_device(labels, ks, w_offset="max+1", one_pass=False)
        assert got[3] == want[3]
        for x, y in zip(got[:3], want[:3]):
            assert torch.equal(x, y)
