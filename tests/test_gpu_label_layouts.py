"""The MFMA labeling at the edges of its layouts (packed and split rows,
partial groups and tiles, point blocks past the end, scales) and its
cascade, against the FP64 direct labeling, which equals the oracle
(MyML/MyML/cluster/KMeans.py:453-490): the same labels and distances."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


def _same(torch, X, C, ks=None):
    from masters_final_amd.cluster.KMeans import label_device
    a, da, nres = label_device(X, C, k_list=ks, precision="bf16x3")
    b, db, _ = label_device(X, C, k_list=ks, precision="fp64")
    assert torch.equal(a, b) and torch.equal(da, db)
    return nres


@pytest.mark.parametrize("d", [4, 5, 10, 11, 15, 16, 21, 22, 32, 33, 42, 43, 53, 54, 64, 65, 74, 75,
                               85, 86, 97, 127, 128])
@pytest.mark.parametrize("n,ks", [(1, [700]), (257, [1, 2, 5, 63, 64, 65, 1500]), (4100, [901])])
def test_every_layout_equals_fp64(torch, d, n, ks):
    g = torch.Generator(device="cuda").manual_seed(d * 1000 + n)
    X = torch.randn((n, d), generator=g, device="cuda") * 3
    C = torch.randn((sum(ks), d), generator=g, device="cuda") * 3
    C[::7] = X[torch.arange(C[::7].shape[0], device="cuda") % n]  # exact hits
    _same(torch, X, C, ks)


@pytest.mark.parametrize("sx,sc", [(1e-18, 1e-18), (1e15, 1e15), (1.0, 1e9), (1e9, 1.0), (0.0, 1.0)])
def test_scales_equal_fp64(torch, sx, sc):
    g = torch.Generator(device="cuda").manual_seed(3)
    X = torch.randn((1000, 24), generator=g, device="cuda") * sx
    C = torch.randn((300, 24), generator=g, device="cuda") * sc
    X[5] *= 1e-6  # a row far below its block's scale
    C[7] *= 1e-6
    _same(torch, X, C)


@pytest.mark.parametrize("d,k", [(40, 2600), (64, 1300), (100, 700)])
@pytest.mark.parametrize("ties", [False, True])
def test_cascade_equals_fp64(torch, d, k, ties):
    """Large enough for the cascade; ties: every centroid twice, so the single
    product certifies nothing and the sample sends all rows to the three
    products (and then to the re-scoring of many flags)."""
    n = 240_001 if d < 100 else 200_003
    g = torch.Generator(device="cuda").manual_seed(k)
    m = torch.randn((50, d), generator=g, device="cuda") * 2
    X = torch.randn((n, d), generator=g, device="cuda")
    X += m[torch.randint(0, 50, (n,), generator=g, device="cuda")]
    C = X[torch.randperm(n, generator=g, device="cuda")[:k]].clone()
    if ties:
        C[k // 2:k // 2 * 2] = C[:k // 2]
    assert n * k * ((d + 31) // 32) >= 5e8
    nres = _same(torch, X, C)
    assert (nres > n // 2) == ties


@pytest.mark.parametrize("n", [255, 256, 257, 511, 512, 513, 2570])
@pytest.mark.parametrize("d", [1, 2, 3, 4])
def test_direct_points_per_lane(torch, n, d):
    """The FP64 form with one and with two points a lane (enough partitions):
    the same labels and distances, bit for bit, NaN rows included."""
    from masters_final_amd.cluster.KMeans import label_device
    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d)).astype(np.float32)
    X[n // 2] = np.nan
    C = rng.standard_normal((5, d)).astype(np.float32)
    a, da, _ = label_device(X, C, precision="fp64")
    P = 600
    b, db, _ = label_device(X, np.tile(C, (P, 1)), [5] * P, precision="fp64")
    assert torch.equal(b, a.expand(P, n))
    assert torch.equal(db.view(torch.int32), da.expand(P, n).contiguous().view(torch.int32))
    with np.errstate(invalid="ignore"):
        D = ((X[:, None].astype(np.float64) - C[None].astype(np.float64)) ** 2).sum(-1)
    want = np.where(np.isnan(D).any(1), 0, D.argmin(1))
    assert np.array_equal(a[0].cpu().numpy(), want)


@pytest.mark.parametrize("d", [1, 2, 3, 4, 7, 8, 16, 17])
@pytest.mark.parametrize("k", [1, 3, 4, 5, 8, 127, 128, 255, 256, 257, 515])
@pytest.mark.parametrize("P", [1, 300])
def test_direct_fours(torch, d, k, P):
    """The plain labeling's groups of four at the edges of groups and of
    centroid tiles, with one and with two points a lane: ties go to the lowest
    index, NaN centroids lose unless they come first, in the oracle's FP64
    arithmetic (ascending dimensions, strict <)."""
    from masters_final_amd.cluster.KMeans import label_device
    rng = np.random.default_rng(1000 * d + k)
    n = 600 if P > 1 else 517
    X = rng.integers(-3, 4, (n, d)).astype(np.float32)  # coarse: many equal distances
    C = rng.integers(-3, 4, (k, d)).astype(np.float32)
    X[5], X[6] = 1e30, np.nan
    if k > 4:
        C[3], C[k - 1] = np.nan, np.inf
    got, dist, _ = label_device(X, np.tile(C, (P, 1)), [k] * P, precision="fp64")
    f32, _, _ = label_device(X, np.tile(C, (P, 1)), [k] * P, precision="fp32")
    D = np.zeros((n, k))
    with np.errstate(all="ignore"):
        for j in range(d):
            t = X[:, j, None].astype(np.float64) - C[None, :, j].astype(np.float64)
            D = D + t * t
    want = np.where(np.isnan(D[:, 0]), 0, np.where(np.isnan(D), np.inf, D).argmin(1))
    assert np.array_equal(got.cpu().numpy(), np.broadcast_to(want, (P, n)))
    ref = D[np.arange(n), want].astype(np.float32)
    assert np.array_equal(dist.cpu().numpy(), np.broadcast_to(ref, (P, n)), equal_nan=True)
    small = np.ones(n, bool)
    small[5] = False  # whose squares leave float32's range
    assert np.array_equal(f32.cpu().numpy()[:, small], np.broadcast_to(want[small], (P, n - 1)))
