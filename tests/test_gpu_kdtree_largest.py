"""A tree of 2^30 - 1 points in two dimensions: the presort's positions go up to
2^31 - 3, within a workgroup's stride of the largest 32-bit integer.  One level
(leaves of 2^29 points): the points must come out in the stable order of their
wider coordinate.  Needs 170 GB of device memory, most of it for a moment."""
import gc

import pytest

import hmx

pytestmark = pytest.mark.gpu


def test_positions_up_to_the_largest_integer():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    gc.collect()
    torch.cuda.empty_cache()
    ctx = hmx.Context()
    hmx.memory_release(ctx)
    if torch.cuda.mem_get_info()[0] < 170 << 30:
        pytest.skip("170 GB of free device memory")
    n = (1 << 30) - 1
    g = torch.Generator(device="cuda").manual_seed(1)
    p = torch.rand(2 * n, generator=g, dtype=torch.float64, device="cuda")
    p[:n].mul_(2.0)
    p[:n:1000] = 0.5  # ties
    tree = hmx.constructKDTree(ctx, n, 2, 1 << 29, p)
    hmx.memory_release(ctx)
    assert tree.info()[2] == 1
    x = tree.reorder(ctx, p[:n], False)
    idx = tree.reorder(ctx, torch.arange(n, dtype=torch.float64, device="cuda"), False)
    asc = x[1:] > x[:-1]
    asc |= (x[1:] == x[:-1]) & (idx[1:] > idx[:-1])
    assert bool(asc.all())
    idx = idx.long()
    assert torch.equal(p[:n][idx], x)
    seen = torch.zeros(n, dtype=torch.bool, device="cuda")
    seen[idx] = True
    assert bool(seen.all())
    del tree, x, idx, asc, seen, p
    torch.cuda.empty_cache()
    hmx.memory_release(ctx)
