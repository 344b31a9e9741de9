"""Passes of 16, 32, 48 and 64 right-hand sides on the matrix cores: a call
of any width gives each column what a call of 16 gives it.

Every column is summed in the same order whatever the pass width, so FP64
columns are equal bit for bit; mixed ones too (the right-hand sides' scales
are per column).  Widths at and around the pass widths, and alternating
widths on one plan (the workspaces' layout depends on the width).
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


@pytest.fixture(scope="module", params=[(4096, 2, 32), (5001, 3, 64)], ids=["full-2d-b32", "partial-3d-b64"])
def pipe(request, torch_cuda):
    n, d, b = request.param
    pp = hmx.Pipeline(n, d, b, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL,
                      points=to_dev(torch_cuda, O.generate_points(n, d, 7)), direct=True)
    pp.make_mixed(3e-6)
    return pp


@pytest.mark.parametrize("mixed", [False, True], ids=["fp64", "mixed"])
@pytest.mark.parametrize("layout", [1, 2], ids=["in-place", "copied"])
def test_any_width_equals_passes_of_16(torch_cuda, pipe, mixed, layout):
    torch = torch_cuda
    if mixed and layout == 1:
        pytest.skip("the mixed plan has one layout")
    pipe.H.set_fp64_layout(layout)
    g = torch.Generator(device="cuda").manual_seed(3)
    X = torch.randn(130, pipe.n, generator=g, device="cuda", dtype=torch.float32 if mixed else torch.float64)
    f = pipe.matvec_mixed if mixed else pipe.matvec
    ref = torch.cat([f(X[a:a + 16].contiguous()) for a in range(0, 128, 16)] + [f(X[128:].contiguous())])
    for k in (17, 64, 31, 32, 33, 2, 48, 49, 65, 100, 130, 16):
        assert torch.equal(f(X[:k].contiguous()), ref[:k]), k
