"""The library's held memory and stream captures.

  * A build in one thread, allocating and freeing all the time, does not
    disturb a capture that another thread has open (thread-local mode, the one
    batched products use), and is not disturbed by it.
  * A call that would have to allocate inside its own capture is refused, as
    hipMalloc refuses it, also when a held block of the right size is at hand:
    the graph would keep addresses that a later call may give away.
"""
import ctypes
import threading

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


def make(torch, ctx, n, d, b):
    return hmx.Pipeline(n, d, b, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL,
                        points=to_dev(torch, O.generate_points(n, d, 13)), ctx=ctx, direct=True)


def test_a_build_beside_another_threads_capture(torch_cuda):
    torch = torch_cuda
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx = hmx.Context(s)
        x = to_dev(torch, O.generate_rhs(3000, 4, 3).T)
        pts = to_dev(torch, O.generate_points(3000, 2, 13))
        s.synchronize()

        def build():
            p = hmx.Pipeline(3000, 2, 32, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL, points=pts, ctx=ctx,
                             direct=True)
            return p.matvec(x)

        ref = build()
        s.synchronize()
        opened, finish, errors, replayed = threading.Event(), threading.Event(), [], []

        def capture():
            try:
                own = torch.cuda.Stream()
                with torch.cuda.stream(own):
                    a = torch.zeros(1000, device="cuda")
                    own.synchronize()
                    g = torch.cuda.CUDAGraph()
                    g.capture_begin(capture_error_mode="thread_local")
                    try:
                        a.add_(1.0)
                        opened.set()
                        finish.wait(60)
                    finally:
                        g.capture_end()
                    g.replay()
                    g.replay()
                    own.synchronize()
                    replayed.append(a.cpu())
            except Exception as e:  # reported below
                errors.append(e)
                opened.set()

        t = threading.Thread(target=capture)
        t.start()
        try:
            assert opened.wait(60)
            out = []
            with torch.cuda.stream(s):
                # only the library's own calls: torch's allocator stays out of it
                tree = hmx.constructKDTree(ctx, 3000, 2, 32, pts)
                st = hmx.constructHMatrixStructure(ctx, 3000, 2, 32, "maxDiam", 1.0, tree)
                cfg = hmx.default_config(numberOfInputPoints=3000, dimensionOfInputPoints=2, bucketSize=32,
                                         lowestLevelTolerance=1e-6, maxRankPolicy=hmx.MAXRANK_FULL,
                                         admissibilityCondition=hmx.ADMISSIBILITY["maxDiam"])
                for _ in range(3):
                    H = hmx.generateHMatrixDirect(ctx, cfg, tree, st, pts)
                    out.append(H.level_info(H.num_levels - 1)["rankSum"])
                    H.free()
        finally:
            finish.set()
            t.join()
        assert not errors, errors
        assert torch.equal(replayed[0], torch.full((1000,), 2.0))
        assert len(set(out)) == 1
        assert torch.equal(build(), ref)


def test_allocation_inside_a_capture_is_refused(torch_cuda):
    torch = torch_cuda
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx = hmx.Context(s)
        pipe = make(torch, ctx, 3000, 2, 32)
        X = to_dev(torch, O.generate_rhs(3000, 64, 3).T)
        Y = torch.empty_like(X)
        wide = pipe.matvec(X)
        # the wide workspaces go back, the narrow call's allocations wait for the device once
        pipe.H.set_fp64_layout(0)
        x4, y4 = X[:4].contiguous(), torch.empty(4, 3000, dtype=torch.float64, device="cuda")
        ref = pipe.matvec(x4)
        s.synchronize()
        hmx.HMatrixVecMult(ctx, pipe.H, 4, x4, y4)
        s.synchronize()
        hip = hmx.lib()  # the HIP runtime the library is linked with
        stream, graph = ctypes.c_void_p(s.cuda_stream), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local
        try:
            with pytest.raises(hmx.HmxError):
                hmx.HMatrixVecMult(ctx, pipe.H, 64, X, Y)
        finally:
            hip.hipStreamEndCapture(stream, ctypes.byref(graph))  # the refusal ended the capture
            hip.hipGetLastError()
            # the runtime gives the stream back with the next capture's end
            assert hip.hipStreamBeginCapture(stream, 1) == 0
            assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        s.synchronize()
        assert torch.equal(pipe.matvec(x4), ref)
        assert torch.equal(pipe.matvec(X), wide)
