"""A batch whose tuning ran out of memory in the middle of a plan still
multiplies: the half-built plan is not used, the next call builds it.

Bar: 1e-13 of the norm against the product before (the phase-1 chunk length,
and with it the order of the sums, is whatever the tuning had got to)."""
import ctypes

import pytest

import hmx
import oracle as O
from test_gpu_pipeline import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
def test_products_after_a_failed_tuning(graph):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    L = hmx.lib()
    bp = hmx.BatchPipeline([(700, 2, 0.1), (1500, 3, 0.2)], b=32)
    x = to_dev(torch, O.generate_rhs(2200, 1, 3).T)[0].contiguous()
    y = torch.empty_like(x)
    ref = bp.matvec(x, graph=graph).clone()
    norm = float(torch.linalg.norm(ref))
    chunk, ms = ctypes.c_int32(), ctypes.c_float()

    def tune():
        return L.hmx_batch_tune(bp.ctx.handle, bp.batch.handle, 1, ctypes.byref(chunk), ctypes.byref(ms))

    L.hmx_debug_set_alloc_fault(-1)
    assert tune() == hmx.HMX_OK
    total = L.hmx_debug_alloc_count()
    assert total > 10
    for fault in range(total):
        L.hmx_debug_set_alloc_fault(fault)
        try:
            st = tune()
        finally:
            L.hmx_debug_set_alloc_fault(-1)
        assert st in (hmx.HMX_OK, hmx.HMX_ENOMEM), fault
        bp.matvec(x, y, graph=graph)
        torch.cuda.synchronize()
        assert float(torch.linalg.norm(y - ref)) <= 1e-13 * norm, fault
    assert tune() == hmx.HMX_OK
    bp.matvec(x, y, graph=graph)
    assert float(torch.linalg.norm(y - ref)) <= 1e-13 * norm
