"""One graph's cut on both sides of the size where the batch's kernels give way
to the parallel ones, against the oracle's rules."""
import pytest
from test_gpu_cut_batches import test_single_graph_forms as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [49_152, 49_153])
def test_single_graph_at_the_limit(n):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _check(torch, n)
