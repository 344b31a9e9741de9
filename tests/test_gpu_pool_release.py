"""hmx_memory_held / hmx_memory_release on the device: what a freed H-matrix
leaves held is within the stated bound, goes back to the driver when asked, and
products before and after are equal."""
import gc

import pytest

import hmx
import oracle as O
from test_gpu_pipeline import to_dev

pytestmark = pytest.mark.gpu


def test_release_gives_the_held_memory_back():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ctx = hmx.Context()
    n = 16384
    pts = to_dev(torch, O.generate_points(n, 3, 5))
    x = to_dev(torch, O.generate_rhs(n, 5, 2).T)

    def product():
        p = hmx.Pipeline(n, 3, 64, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL, points=pts, ctx=ctx, direct=True)
        return p.matvec(x)

    ref = product()
    gc.collect()
    torch.cuda.synchronize()
    held = hmx.memory_held(ctx)
    free0, total = torch.cuda.mem_get_info()
    print(f"held {held >> 20} MiB, free {free0 >> 20} MiB")
    assert 0 < held <= min(total // 16, (free0 + held) // 8)
    hmx.memory_release(ctx)
    assert hmx.memory_held(ctx) == 0
    assert torch.cuda.mem_get_info()[0] >= free0 + held // 2  # the driver has it again (it may round)
    assert torch.equal(product(), ref)
