"""Centroids and points that hold NaNs in the MFMA labeling, whose re-scoring
must give what the FP64 direct labeling gives, which equals the oracle
(MyML/MyML/cluster/KMeans.py:453-490): a NaN distance never replaces another,
and the first centroid's is never replaced."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.mark.parametrize("n,d,ks", [
    (40, 5, [30, 700]), (300, 16, [70]), (300, 18, [10, 1, 64, 200]), (9000, 37, [300]),
    (9000, 100, [65, 2, 1200]), (2000, 128, [90]), (70_000, 24, [40]), (70_000, 24, [40, 300])])
@pytest.mark.parametrize("which", ["some", "first", "all but one", "points"])
def test_nans_equal_fp64(torch, n, d, ks, which):
    from masters_final_amd.cluster.KMeans import label_device
    g = torch.Generator(device="cuda").manual_seed(n + d)
    X = torch.randn((n, d), generator=g, device="cuda")
    C = torch.randn((sum(ks), d), generator=g, device="cuda")
    at = 0
    for k in ks:
        bad = {"some": slice(at + 1, at + k, 5), "first": slice(at, at + 1),
               "all but one": [at + q for q in range(k) if q != k // 2],
               "points": slice(0, 0)}[which]
        C[bad, d // 2] = float("nan")
        at += k
    if which == "points":
        X[::7, 1] = float("nan")
    a, da, _ = label_device(X, C, k_list=ks, precision="bf16x3")
    b, db, _ = label_device(X, C, k_list=ks, precision="fp64")
    assert torch.equal(a, b)
    assert torch.equal(torch.nan_to_num(da, nan=-1.0), torch.nan_to_num(db, nan=-1.0))
