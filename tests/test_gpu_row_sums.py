"""The workgroup form of numpy's float32 sum (the inertia of
MyML/cluster/KMeans.py:164) at the edges of its leaves, chunks and tails:
numpy's result to the bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.mark.parametrize("sizes", [
    tuple(range(1, 20)) + tuple(range(120, 145)) + tuple(range(250, 275)),
    tuple(range(500, 530)) + tuple(range(1016, 1056)) + (2047, 2049, 2087, 2175),
    (4095, 4096, 4097, 4200, 8063, 8183, 8184, 8190, 8191, 8192, 8193, 8199, 8200, 8320, 8321),
    (16_383, 16_385, 100_003)])
def test_row_sums_equal_numpy(torch, sizes):
    from masters_final_amd.cluster.KMeans import sum_f32_device
    rng = np.random.default_rng(sizes[0])
    for n in sizes:
        # magnitudes apart enough that another order rounds differently
        a = (rng.standard_normal((3, n)) * 10.0 ** rng.integers(-3, 4, (3, n))).astype(np.float32)
        a[2] = np.abs(a[2])
        got = sum_f32_device(torch.from_numpy(a).cuda()).cpu().numpy()
        want = np.array([row.sum() for row in a], dtype=np.float32)
        assert got.tobytes() == want.tobytes(), n


def test_row_sums_of_special_values(torch):
    from masters_final_amd.cluster.KMeans import sum_f32_device
    a = np.zeros((4, 300), np.float32)
    a[0] = -0.0
    a[1, 290] = np.inf
    a[2, 3], a[2, 200] = np.inf, -np.inf
    a[3] = np.float32(3e38)
    got = sum_f32_device(torch.from_numpy(a).cuda()).cpu().numpy()
    with np.errstate(all="ignore"):
        want = np.array([row.sum() for row in a], dtype=np.float32)
    assert np.array_equal(got, want, equal_nan=True)
