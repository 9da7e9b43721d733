"""The default build of mid-sized matrices (one visit, a pool for every pair)
against the two-visit build, at the limits of its range: exactly equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.mark.parametrize("n,P,k,full,path", [
    (4095, 9, 40, False, "two-pass"), (4096, 9, 40, False, "one-pass"),
    (4097, 300, 700, True, "one-pass"), (5000, 6, 1, False, "one-pass"),
    (5000, 3, 1, True, "one-pass"), (16_385, 4, 90, True, "two-pass"),
    (23_170, 4, 300, False, "one-pass"), (23_172, 4, 300, False, "two-pass")])
def test_bound_build(torch, n, P, k, full, path):
    from masters_final_amd.EAC.sparse import coassoc_device
    rng = np.random.default_rng(n + P)
    labels = rng.integers(0, k, (P, n)).astype(np.int32)
    if P > 4:
        labels[1, ::7] = -1  # samples not listed
    ks = [k] * P
    info = {}
    a = coassoc_device(labels, ks, full_rows=full, w_offset="max+1", info=info)
    b = coassoc_device(labels, ks, full_rows=full, w_offset="max+1", one_pass=False)
    assert info["path"] == path
    assert a[3] == b[3]
    for x, y in zip(a[:3], b[:3]):
        assert torch.equal(x, y)


def test_bound_build_reports_bad_labels(torch):
    from masters_final_amd._lib import EACError
    from masters_final_amd.EAC.sparse import coassoc_device
    labels = np.zeros((2, 5000), np.int32)
    labels[1, 4999] = 3
    with pytest.raises(EACError, match="label >= k"):
        coassoc_device(labels, [1, 3])


@pytest.mark.parametrize("fails", [(0,), (1,), (2,)])
def test_bound_build_without_room(torch, monkeypatch, fails):
    """The pool (allocation 0), the columns (1) or the values (2) do not fit
    beside each other: the two visits, which need no pool, take over."""
    from masters_final_amd.EAC.sparse import coassoc_device
    n, P = 5000, 6
    labels = np.random.default_rng(5).integers(0, 40, (P, n)).astype(np.int32)
    want = coassoc_device(labels, [40] * P, w_offset="max+1", one_pass=False)
    dl = torch.from_numpy(labels).cuda()
    empty, seen = torch.empty, []

    def scarce(*a, **kw):
        if kw.get("dtype") in (torch.uint8, torch.int32):
            seen.append(a)
            if len(seen) - 1 in fails:
                raise torch.cuda.OutOfMemoryError("none left")
        return empty(*a, **kw)

    coassoc_device(labels, [40] * P)  # the shared workspace is there
    monkeypatch.setattr(torch, "empty", scarce)
    info = {}
    got = coassoc_device(dl, [40] * P, w_offset="max+1", info=info)
    assert info["path"] == "two-pass" and len(seen) == fails[0] + 3
    assert got[3] == want[3]
    for x, y in zip(got[:3], want[:3]):
        assert torch.equal(x, y)
