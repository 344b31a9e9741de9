"""Infinities and NaN of one product stay out of the next ones, whatever their
widths: z's padding columns lie elsewhere at every pass width, and hold what an
earlier call or nobody left there.  Eagerly, and in a graph captured at one
width and replayed after calls of others (several replays, each against the
eager result)."""
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


@pytest.fixture(scope="module", params=[(4096, 2, 32), (5001, 3, 64)], ids=["full-2d-b32", "partial-3d-b64"])
def setup(request, torch_cuda):
    torch = torch_cuda
    n, d, b = request.param
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx = hmx.Context(s)
        pp = hmx.Pipeline(n, d, b, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL, ctx=ctx,
                          points=to_dev(torch, O.generate_points(n, d, 7)), direct=True)
        pp.make_mixed(3e-6)
        X = to_dev(torch, O.generate_rhs(n, 64, 3).T)
        s.synchronize()
    return s, pp, X


PATHS = [("fp64", 1), ("fp64", 2), ("transposed", 1), ("transposed", 2), ("mixed", 0)]


def product(pp, path, X, Y=None):
    if path == "mixed":
        return pp.matvec_mixed(X, Y)
    return pp.matvec(X, Y, transpose=path == "transposed")


@pytest.mark.parametrize("split", [0, 1], ids=["whole-leaves", "split-leaves"])
@pytest.mark.parametrize("path,layout", PATHS)
@pytest.mark.parametrize("k,other", [(40, 8), (8, 40), (64, 20), (20, 64), (48, 33)])
def test_a_graph_replayed_after_other_widths(torch_cuda, setup, path, layout, k, other, split):
    torch = torch_cuda
    s, pp, X = setup
    assert hmx.lib().hmx_debug_set_wave_split(pp.H.handle, split) == hmx.HMX_OK
    with torch.cuda.stream(s):
        if layout:
            pp.H.set_fp64_layout(layout)
        else:
            pp.make_mixed(3e-6)
        X = X.float() if path == "mixed" else X
        x, bad = X[:k].contiguous(), X[:other].clone()
        bad[0] = float("nan")
        bad[1, ::7] = float("inf")
        product(pp, path, X)  # workspaces of every width
        ref = product(pp, path, x).clone()
        assert bool(torch.isfinite(ref).all())
        y, yb = torch.empty_like(x), torch.empty_like(bad)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s, capture_error_mode="thread_local"):
            product(pp, path, x, y)
        for _ in range(3):
            product(pp, path, bad, yb)
            assert bool(torch.isfinite(yb[2:]).all())  # the other columns of that call
            y.fill_(-1.0)
            g.replay()
            s.synchronize()
            assert torch.equal(y, ref)
            assert torch.equal(product(pp, path, x), ref)
