"""Dense counts of a matrix whose tiles are more than one grid dimension can
number (n > 370,727: 2^32 threads), against the labels themselves (the counts
of MyML/MyML/EAC/full.py:155-166 for one partition)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_counts_of_more_tiles_than_a_grid_dimension_numbers():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from masters_final_amd.EAC.full import coassoc_dense_device
    n = 370_800  # 68.7 GB of one-byte pairs
    if torch.cuda.mem_get_info()[0] < (80 << 30):
        pytest.skip("less than 80 GiB of device memory free")
    lab = (torch.arange(n, device="cuda", dtype=torch.int32) * 7919) % 1000
    out, mx = coassoc_dense_device(lab, condensed=True, dtype=np.uint8)
    assert mx == 1
    for i in (0, 1, 63, 64, 9999, n // 3, n // 2, n - 600, n - 129, n - 2):
        at = n * i - i * (i + 1) // 2
        row = out[at:at + n - 1 - i]
        assert torch.equal(row, (lab[i + 1:] == lab[i]).to(torch.uint8)), i
    del out
    torch.cuda.empty_cache()
