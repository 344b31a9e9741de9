"""The transposed product's matrix-core plan against the transposed dense
expansion of the H-matrix's own factors: dense near-field blocks (U and V of
different tiles exchanged), factors in place and copied, full and partial
leaves, after a change of the factors; widths around the kernels' 16-column
blocks and 64-column passes.

Bar: 1e-13 of the norm, as for the forward product (FP64 sums of at most
4096 terms on both sides).
"""
import numpy as np
import pytest

import hmx
import oracle as O
from test_gpu_pipeline import expand_gpu, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture(scope="module", params=[(4096, 2, 32), (3000, 2, 64), (1111, 3, 32)],
                ids=["full-2d-b32", "partial-2d-b64", "partial-3d-b32"])
def pipe(request, torch_cuda):
    n, d, b = request.param
    p = O.generate_points(n, d, 29)
    pp = hmx.Pipeline(n, d, b, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL, points=to_dev(torch_cuda, p),
                      direct=True)
    # tiles compressed on their own: (u, v) and (v, u) are not transposes
    pp.E = expand_gpu(pp.ctx, pp)
    return pp


@pytest.mark.parametrize("layout", [1, 2], ids=["in-place", "copied"])
@pytest.mark.parametrize("k", [2, 16, 17, 64, 65])
def test_transposed_plan(torch_cuda, pipe, k, layout):
    pipe.H.set_fp64_layout(layout)
    X = O.generate_rhs(pipe.n, k, 3 + k)
    y = pipe.matvec(to_dev(torch_cuda, X.T), transpose=True).cpu().numpy().T
    ref = pipe.E.T @ X
    assert np.linalg.norm(y - ref) / np.linalg.norm(ref) < 1e-13


def test_transposed_plan_follows_the_factors(torch_cuda, pipe):
    torch = torch_cuda
    level = next(l for l in range(1, pipe.H.num_levels) if pipe.H.level_info(l)["rankSum"])
    pipe.H.set_fp64_layout(2)
    x = to_dev(torch_cuda, O.generate_rhs(pipe.n, 4, 5).T)
    before = pipe.matvec(x, transpose=True)
    u, v = pipe.H.level_device(pipe.ctx, level)
    hmx._check(hmx.lib().hmx_hmatrix_set_level(pipe.ctx.handle, pipe.H.handle, level, hmx._ptr(2.0 * u), hmx._ptr(v)))
    twice = pipe.matvec(x, transpose=True)
    hmx._check(hmx.lib().hmx_hmatrix_set_level(pipe.ctx.handle, pipe.H.handle, level, hmx._ptr(u), hmx._ptr(v)))
    assert torch.equal(pipe.matvec(x, transpose=True), before)
    assert not torch.equal(twice, before)
