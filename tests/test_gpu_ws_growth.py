"""A workspace growth that runs out of memory leaves nothing behind: the call
that needed it fails with HMX_ENOMEM (or gets by with less memory and gives the
right answer), and calls of the former width go on giving what they gave.

Every allocation that the wider call makes is failed in turn (the allocation
counter's test hook), on partial leaves, where the vectors are copied too.
"""
import ctypes

import pytest

import hmx
import oracle as O
from test_gpu_pipeline import to_dev

pytestmark = pytest.mark.gpu

N, D, B = 1111, 3, 32  # partial leaves


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture(scope="module")
def pipe(torch_cuda):
    return hmx.Pipeline(N, D, B, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL,
                        points=to_dev(torch_cuda, O.generate_points(N, D, 11)), direct=True)


def grads(torch, pipe, x, w):
    """Factor gradients of all levels, one after the other."""
    H, L = pipe.H, pipe.H.num_levels - 1
    size = {l: H.level_info(l)["rankSum"] * (1 << (L - l)) * B for l in range(1, L + 1)}
    dU = {l: torch.empty(size[l], dtype=torch.float64, device="cuda") for l in size if size[l]}
    dV = {l: torch.empty_like(dU[l]) for l in dU}
    pu = (ctypes.c_void_p * L)(*[dU[l].data_ptr() if l in dU else 0 for l in range(1, L + 1)])
    pv = (ctypes.c_void_p * L)(*[dV[l].data_ptr() if l in dV else 0 for l in range(1, L + 1)])
    hmx._check(hmx.lib().hmx_hmatvec_grad_factors(pipe.ctx.handle, H.handle, x.shape[0], hmx._ptr(x), hmx._ptr(w), pu, pv),
               pipe.ctx)
    return torch.cat([t for l in dU for t in (dU[l], dV[l])])


def profile(torch, pipe, x):
    """The streaming kernels with several right-hand sides."""
    y = torch.empty_like(x)
    hmx.matvec_profile(pipe.ctx, pipe.H, x.shape[0], x, y, iters=1)
    return y


@pytest.mark.parametrize("path", ["forward", "transposed", "mixed", "gradients", "streaming", "batch"])
def test_a_failed_growth_leaves_narrow_calls_working(torch_cuda, pipe, path):
    torch, L = torch_cuda, hmx.lib()
    g = torch.Generator(device="cuda").manual_seed(4)
    X = torch.randn(64, N, generator=g, device="cuda", dtype=torch.float32 if path == "mixed" else torch.float64)
    W = torch.randn(64, N, generator=g, device="cuda", dtype=torch.float64)
    obj = pipe
    if path == "batch":
        obj = hmx.BatchPipeline([(700, 2, 0.1), (N, 3, 0.2)], b=B)
        X = torch.randn(64, 700 + N, generator=g, device="cuda", dtype=torch.float64)

    def call(k):
        x = X[:k].contiguous()
        if path == "gradients":
            return grads(torch, pipe, x, W[:k].contiguous())
        if path == "streaming":
            return profile(torch, pipe, x)
        if path == "mixed":
            return pipe.matvec_mixed(x)
        if path == "batch":
            return obj.matvec(x)
        return pipe.matvec(x, transpose=path == "transposed")

    narrow, wide = (4, 16) if path == "streaming" else (16, 64)
    if path == "mixed":
        pipe.make_mixed(3e-6)
    else:
        pipe.H.set_fp64_layout(0)  # the plans and their workspaces start anew
        pipe.H.set_plan_options(True, True, True)
    ref = call(narrow)
    done = False
    for fault in range(16):
        L.hmx_debug_set_alloc_fault(fault)
        out = None
        try:
            out = call(wide)
            done = L.hmx_debug_alloc_count() <= fault  # no allocation was failed
        except hmx.HmxError as e:
            assert e.status == hmx.HMX_ENOMEM, e
        finally:
            L.hmx_debug_set_alloc_fault(-1)
        torch.cuda.synchronize()
        assert torch.equal(call(narrow), ref), fault
        if out is not None and path != "gradients":
            assert torch.equal(out[:narrow], ref), fault
        if done:
            break
    assert done, "the wide call never got all of its allocations"
    if path != "gradients":
        assert torch.equal(call(wide)[:narrow], ref)
