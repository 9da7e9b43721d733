"""Rows far above the rest of their workgroup in the MFMA labeling: a fill
value or a heavy tail must change no other row's label, and must not send the
other rows to the re-scoring. Against the FP64 direct labeling, which equals
the oracle (MyML/MyML/cluster/KMeans.py:453-490): the same labels and
distances."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


def _data(torch, n, d, ktot, small, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn((n, d), generator=g, device="cuda") * small,
            torch.randn((ktot, d), generator=g, device="cuda") * small)


def _same(torch, X, C, ks=None):
    from masters_final_amd.cluster.KMeans import label_device
    a, da, nres = label_device(X, C, k_list=ks, precision="bf16x3")
    b, db, _ = label_device(X, C, k_list=ks, precision="fp64")
    assert torch.equal(a, b) and torch.equal(da, db)
    return nres


@pytest.mark.parametrize("big,small", [(1e30, 1e-6), (1e30, 1e-5), (1e30, 1e-4), (1e20, 1e-9),
                                       (1e18, 1e-10), (3e38, 1e-6), (float("inf"), 1e-3)])
@pytest.mark.parametrize("n,d,ks", [
    (256, 24, [300]),             # packed rows, one partition
    (400, 16, [40, 200, 7]),      # several partitions
    (300, 64, [500]),             # split rows
    (130_000, 64, [2048]),        # the cascade's single and listed products
])
def test_rows_beside_an_outlier_equal_fp64(torch, n, d, ks, big, small):
    X, C = _data(torch, n, d, sum(ks), small, d + n)
    X[77::1000, 3] = big
    _same(torch, X, C, ks)


@pytest.mark.parametrize("n,d,ks", [(4096, 24, [300]), (4096, 16, [40, 200, 7]),
                                    (130_000, 64, [2048])])
@pytest.mark.parametrize("up", [20, 40])
def test_an_outlier_costs_only_itself(torch, n, d, ks, up):
    """One row in 128 far above the others: without a scale of their own the
    others lose bits and are all scored again in FP64 (n of them); with it
    about one in a hundred is, as beside ordinary rows."""
    X, C = _data(torch, n, d, sum(ks), 1.0, d)
    X[5::128] *= 2.0 ** up
    nres = _same(torch, X, C, ks)
    assert nres <= len(ks) * (X[5::128].shape[0] + n // 20)


@pytest.mark.parametrize("n,d,ks", [(5000, 24, [300]), (5000, 16, [40, 200, 7]),
                                    (130_000, 64, [2048])])
@pytest.mark.parametrize("span", [12, 60, 120])
def test_rows_of_any_scale_equal_fp64(torch, n, d, ks, span):
    """Every row and every centroid at a power of two of its own."""
    X, C = _data(torch, n, d, sum(ks), 1.0, span)
    g = torch.Generator(device="cuda").manual_seed(span)
    X *= 2.0 ** torch.randint(-span, span + 1, (n, 1), generator=g, device="cuda")
    C *= 2.0 ** torch.randint(-span, span + 1, (sum(ks), 1), generator=g, device="cuda")
    _same(torch, X, C, ks)
