"""Products where the device has no memory for the widest passes or for a
second plan: the narrower passes and the streaming kernels do them, and the
answers stay right.  Memory is made to run out with the allocation-failure
hook, one allocation at a time.

Bars: bit equality where only the pass width changes (every column is summed
in the same order), 1e-13 of the norm between the matrix cores and the
streaming kernels (FP64 sums of at most 4096 terms on both sides).
"""
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


@pytest.fixture(scope="module", params=[(4096, 2, 32), (1111, 3, 64)], ids=["full-2d-b32", "partial-3d-b64"])
def pipe(request, torch_cuda):
    n, d, b = request.param
    return hmx.Pipeline(n, d, b, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL,
                        points=to_dev(torch_cuda, O.generate_points(n, d, 19)), direct=True)


def failing(fault, f):
    """f() with allocation number fault failed: (result, whether it was reached)"""
    L = hmx.lib()
    L.hmx_debug_set_alloc_fault(fault)
    try:
        out = f()
        return out, L.hmx_debug_alloc_count() > fault
    finally:
        L.hmx_debug_set_alloc_fault(-1)


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
def test_narrower_passes(torch_cuda, pipe, mixed):
    torch = torch_cuda
    X = to_dev(torch, O.generate_rhs(pipe.n, 130, 3).T)
    X = X.float() if mixed else X

    def renew():
        pipe.H.set_fp64_layout(0)
        if mixed:
            pipe.make_mixed(3e-6)

    f = pipe.matvec_mixed if mixed else pipe.matvec
    renew()
    ref = f(X)
    for fault in range(12):
        renew()
        f(X[:2].contiguous())
        out, reached = failing(fault, lambda: f(X))
        assert torch.equal(out, ref), fault
        for k in (40, 64, 17, 130):  # as wide as the plan now goes
            assert torch.equal(f(X[:k].contiguous()), ref[:k]), (fault, k)
        if not reached:
            break
    assert fault >= 3 and not reached


def test_transposed_without_room_for_its_plan(torch_cuda, pipe):
    torch = torch_cuda
    X = to_dev(torch, O.generate_rhs(pipe.n, 21, 4).T)
    pipe.H.set_fp64_layout(0)
    ref = pipe.matvec(X, transpose=True)
    norm = float(torch.linalg.norm(ref))
    streaming = 0
    for fault in range(64):
        pipe.H.set_fp64_layout(0)  # a new transposed plan
        out, reached = failing(fault, lambda: pipe.matvec(X, transpose=True))
        assert float(torch.linalg.norm(out - ref)) <= 1e-13 * norm, fault
        streaming += not torch.equal(out, ref)
        again = pipe.matvec(X, transpose=True)
        assert torch.equal(again, out), fault
        if not reached:
            break
    assert not reached and streaming > 0
    pipe.H.set_fp64_layout(0)
    assert torch.equal(pipe.matvec(X, transpose=True), ref)
