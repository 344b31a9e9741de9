"""Box slots that no level of a tree fills -- the leaf level's, and those of
segments a POWER_OF_TWO_ON_LEFT tree does not have -- read as zero, whatever
the library's memory held before: another tree's boxes are left behind first."""
import numpy as np
import pytest

import hmx
import oracle as O
from test_gpu_pipeline import to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture(scope="module")
def ctx(torch_cuda):
    return hmx.Context()


@pytest.mark.parametrize("div", [hmx.FULL_TREE, hmx.POWER_OF_TWO_ON_LEFT], ids=["full", "power-of-two"])
@pytest.mark.parametrize("n,d,b", [(10, 2, 32), (1000, 2, 32), (5000, 3, 64), (20000, 3, 32)])
def test_unfilled_slots_are_zero(torch_cuda, ctx, n, d, b, div):
    # boxes of a finer tree on shifted points, twice, so that what is reused is full of them
    p = O.generate_points(n, d, 5)
    for _ in range(2):
        old = hmx.constructKDTree(ctx, n, d, max(1, b // 2), to_dev(torch_cuda, p + 7.0), divMethod=div)
        big = hmx.constructKDTree(ctx, 16 * n, d, b, to_dev(torch_cuda, O.generate_points(16 * n, d, 6) + 7.0),
                                  divMethod=div)
        del old, big
    tree = hmx.constructKDTree(ctx, n, d, b, to_dev(torch_cuda, p), divMethod=div)
    _, _, lo, hi = tree.copy(ctx, n, d)
    levels = tree.info()[2]
    for level in range(levels + 1):
        a, cnt = (1 << level) - 1, 1 << level
        if level == levels:
            cnt = 0  # leaves have no boxes
        elif div == hmx.POWER_OF_TWO_ON_LEFT:
            size = (1 << (n - 1).bit_length()) >> level
            cnt = -(-n // size)
        end = (2 << level) - 1
        assert np.all(hi[a:a + cnt] > lo[a:a + cnt]), level
        assert not lo[a + cnt:end].any() and not hi[a + cnt:end].any(), level
