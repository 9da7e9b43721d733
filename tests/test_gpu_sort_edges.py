"""The radix sort at the edges of its forms (placement by rank, the tile
sizes), exactly, against NumPy's stable sort."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.mark.parametrize("begin,end", [(0, 64), (0, 7), (3, 29), (8, 40), (57, 64), (0, 0)])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1025, 6324, 6325, 12_649, 16_384, 16_385,
                               131_072, 131_073, 262_145, 524_289, 1_048_577])
def test_sort_stable(torch, n, begin, end):
    from masters_final_amd import _lib as L
    lib = L.load_library()
    rng = np.random.default_rng(n + end)
    keys = rng.integers(0, 2**64, n, dtype=np.uint64, endpoint=False)
    keys[n // 2:] &= np.uint64(0x0303030303030303)  # equal digits, equal keys
    keys[n // 3: n // 2] = np.uint64(2**64 - 1)
    vals = np.arange(n, dtype=np.uint32)
    dk = torch.from_numpy(keys.view(np.int64)).cuda()
    dv = torch.from_numpy(vals.view(np.int32)).cuda()
    ok, ov, only = torch.empty_like(dk), torch.empty_like(dv), torch.empty_like(dk)
    ws = L.workspace(lib.eac_sort_workspace_bytes(n, 8, 4))
    L.check(lib.eac_radix_sort_u64(L.ptr(dk), L.ptr(ok), L.ptr(dv), L.ptr(ov), n, begin, end,
                                   L.ptr(ws), ws.numel(), L.stream_ptr()))
    L.check(lib.eac_radix_sort_u64(L.ptr(dk), L.ptr(only), None, None, n, begin, end,
                                   L.ptr(ws), ws.numel(), L.stream_ptr()))
    # whole digits: the last one may reach past the range
    top = min(64, begin + (end - begin + 7) // 8 * 8)
    word = (keys >> np.uint64(begin)) & np.uint64((1 << (top - begin)) - 1) if top > begin \
        else np.zeros(n, np.uint64)
    order = np.argsort(word, kind="stable")
    assert np.array_equal(ok.cpu().numpy().view(np.uint64), keys[order])
    assert np.array_equal(ov.cpu().numpy().view(np.uint32), vals[order])
    assert np.array_equal(only.cpu().numpy().view(np.uint64), keys[order])
