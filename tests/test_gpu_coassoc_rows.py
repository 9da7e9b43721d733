"""The co-association row kernel at the edges of its layouts: byte counters
(up to 255 partitions, a count of exactly 255) and 16-bit ones (256 and
more), windows that are no multiple of a 16-byte counter group, short runs
(flattened through the bitmap) and long ones (walked per wavefront), against
the oracle's exact matrix (MyML/MyML/EAC/sparse.py:154-225)."""
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


def _build(labels, ks, **kw):
    from masters_final_amd.EAC.sparse import coassoc_device
    ip, ind, dat, mx = coassoc_device(labels, ks, **kw)
    return ip.cpu().numpy(), ind.cpu().numpy(), dat.cpu().numpy(), mx


@pytest.mark.parametrize("n,P,kmin,kmax,window", [
    (1100, 5, 1, 2, 0),       # one cluster a partition: every run is long
    (1100, 5, 1, 3, 1002),    # ... and a window of 62.6 counter groups
    (2051, 70, 2, 9, 514),    # around the bitmap's 128 members a partition
    (700, 255, 1, 2, 0),      # every count is 255
    (700, 256, 1, 2, 0),      # every count is 256: 16-bit counters
    (900, 300, 20, 60, 130),  # 16-bit counters, short runs, odd windows
    (65, 64, 3, 30, 64),      # two windows, the last of one column
    (4097, 2, 700, 900, 0),   # almost no pairs
])
@pytest.mark.parametrize("one_pass", [False, True])
def test_row_layouts_equal_the_oracle(torch, n, P, kmin, kmax, window, one_pass):
    from masters_final_amd.tune import get_knobs, set_knobs
    rng = np.random.default_rng(n + P)
    ks = rng.integers(kmin, kmax, P)
    labels = np.stack([rng.integers(0, k, n) for k in ks]).astype(np.int32)
    if kmax > 2:
        labels[rng.integers(0, P, n // 7), rng.integers(0, n, n // 7)] = -1
    saved = get_knobs()
    try:
        set_knobs(co_window=window)
        gi, gc, gd, mx = _build(labels, ks, one_pass=one_pass, sample_stride=3)
        fi, fc, fd, fm = _build(labels, ks, one_pass=one_pass, full_rows=True, sample_stride=3)
    finally:
        set_knobs(**saved)
    ip, ind, cnt = O.coassoc_condensed(labels, ks)
    assert np.array_equal(gi, ip) and np.array_equal(gc, ind) and np.array_equal(gd, cnt)
    assert mx == fm == (int(cnt.max()) if cnt.size else 0)
    # full rows: the same matrix mirrored, rows sorted by column, no diagonal
    rows = np.repeat(np.arange(n), np.diff(ip))
    key = np.concatenate([rows * n + ind, ind.astype(np.int64) * n + rows])
    at = np.argsort(key)
    frow = np.repeat(np.arange(n), np.diff(fi))
    assert np.array_equal(frow * n + fc, key[at])
    assert np.array_equal(fd, np.concatenate([cnt, cnt])[at])
