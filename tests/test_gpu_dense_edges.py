"""Dense small-n path at the edges of its kernels: label ranges of the packed
and the plain comparison, sizes around the tile, piece, merge, sort and
union-find limits, rows that start on any byte.

Single linkage is checked in closed form: with p a permutation of 0..n-1 and
w(i, j) = bit length of p[i] ^ p[j], the clusters at height h are the blocks
p >> h, and Borůvka needs a round for every bit. All values are integers:
every comparison is exact."""
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


def _counts_small_workspace(torch, lab, condensed):
    """The smallest workspace: the tiles transpose the labels themselves."""
    from masters_final_amd import _lib as L
    P, n = lab.shape
    d = torch.from_numpy(lab).cuda()
    out = torch.full((n * (n - 1) // 2,) if condensed else (n, n), 7, dtype=torch.int32,
                     device="cuda")
    ws = torch.empty(256, dtype=torch.uint8, device="cuda")
    L.check(L.load_library().eac_coassoc_dense(L.ptr(d), n, P, 1 if condensed else 0, L.W_I32,
                                               L.ptr(out), None, L.ptr(ws), 256, L.stream_ptr()))
    return out


@pytest.mark.parametrize("condensed", [True, False])
@pytest.mark.parametrize("k", [1, 126, 127, 254, 255, 700])
@pytest.mark.parametrize("n,P", [(2, 1), (63, 3), (64, 32), (65, 33), (131, 70)])
def test_counts_and_sums(torch, n, P, k, condensed):
    from masters_final_amd.EAC.full import EAC_FULL, coassoc_dense_device
    rng = np.random.default_rng(n * 1000 + k)
    lab = rng.integers(max(0, k - 4), k, (P, n)).astype(np.int32)
    if k == 700:
        lab[::2] *= 3_000_000  # labels of 31 bits
    lab[rng.random((P, n)) < 0.1] = -1
    want = O.coassoc_full(lab, condensed=condensed)
    small = _counts_small_workspace(torch, lab, condensed)
    assert np.array_equal(small.cpu().numpy(), want)
    for dtype in (np.uint8, np.uint16, np.int32, np.float32):
        got, mx = coassoc_dense_device(lab, condensed=condensed, dtype=dtype)
        assert np.array_equal(got.cpu().numpy().astype(np.int64), want) and mx == want.max()
        if dtype == np.uint16:
            continue
        m = EAC_FULL(n, dtype=dtype, condensed=condensed)
        for _ in range(4):  # 4 x 70 wraps in uint8
            m.update_labels(lab)
        four = 4 * want if dtype != np.uint8 else (4 * want) % 256
        assert np.array_equal(m.coassoc.cpu().numpy().astype(np.int64), four)


@pytest.mark.parametrize("dtype", [np.uint8, np.int32, np.float32])
@pytest.mark.parametrize("off", [0, 1, 3])
def test_degree_and_diassoc_any_start(torch, dtype, off):
    from masters_final_amd.EAC.full import EAC_FULL
    rng = np.random.default_rng(off)
    for n in (1, 2, 5, 77, 1000):
        for condensed in (True, False):
            size = n * (n - 1) // 2 if condensed else n * n
            if not size:
                continue
            a = (rng.integers(0, 90, size) * (rng.random(size) < 0.4)).astype(dtype)
            buf = torch.zeros(size + off, dtype=torch.from_numpy(a).dtype, device="cuda")
            buf[off:] = torch.from_numpy(a).cuda()
            m = EAC_FULL(n, dtype=dtype, condensed=condensed)
            m.coassoc = buf[off:] if condensed else buf[off:].view(n, n)
            m.get_degree()
            sq = np.zeros((n, n), dtype)
            if condensed:
                sq[np.triu_indices(n, 1)] = a
            else:
                sq = a.reshape(n, n)
            assert np.array_equal(m.degree, (sq != 0).sum(1)) and m.nnz == int((a != 0).sum())
            m.make_diassoc()
            assert np.array_equal(m.coassoc.cpu().numpy().ravel().astype(np.int64),
                                  int(a.max()) + 1 - a.astype(np.int64))
            assert not buf[:off].any()


def _bit_matrix(torch, p, condensed, dtype):
    n = p.numel()
    cols = torch.arange(n, device="cuda")
    parts = []
    for r0 in range(0, n, 1024):
        r = cols[r0:r0 + 1024]
        x = (p[r][:, None] ^ p[None, :]).double()
        w = torch.where(x > 0, torch.floor(torch.log2(x.clamp(min=1))) + 1, x).to(torch.int32)
        parts.append(w[cols[None, :] > r[:, None]].to(dtype) if condensed else w.to(dtype))
    return torch.cat(parts)


@pytest.mark.parametrize("n,dtype,condensed", [
    (2, "uint8", True), (3, "uint8", False), (17, "float32", True), (17, "int32", False),
    (63, "uint8", True), (64, "uint16", False), (65, "uint8", False), (130, "uint16", True),
    (1000, "uint8", True), (1001, "uint8", False), (1003, "float32", False),
    (1025, "int32", True), (12288, "uint8", True), (12289, "uint8", False),
    (16384, "uint8", True), (16385, "uint16", True), (32768, "uint8", True),
    (32769, "uint8", True)])
def test_single_linkage_closed_form(torch, n, dtype, condensed):
    from masters_final_amd.EAC.full import full_sl_lifetime_device
    perm = np.random.default_rng(n).permutation(n)
    p = torch.from_numpy(perm).cuda()
    m = _bit_matrix(torch, p, condensed, getattr(torch, dtype))
    bits = int(n - 1).bit_length()
    blocks = [((n - 1) >> h) + 1 for h in range(bits + 1)]  # clusters at height h
    for h in range(bits):
        want_Z = n <= 12289 and h == 0
        nc, lab, Z = full_sl_lifetime_device(m, n, n_clusters=blocks[h], want_Z=want_Z)
        first = {}
        want = np.array([first.setdefault(b, len(first)) for b in (perm >> h).tolist()])
        assert nc == blocks[h]
        if lab is None:
            assert nc == 1
        else:
            assert np.array_equal(lab.cpu().numpy(), want)
        if Z is not None:
            heights = np.repeat(np.arange(1, bits + 1),
                                [blocks[g] - blocks[g + 1] for g in range(bits)])
            assert np.array_equal(Z[:, 2].cpu().numpy(), heights)
            assert Z[-1, 3].item() == n
