"""The two splits of the matrix-core products' work over waves -- 64 columns of
an item and a whole leaf per wave, as in large plans, or 16 columns and 16 rows,
as in small ones -- on the same H-matrices: bit for bit equal (the same sums in
the same order), and FP64 products within 1e-13 of the dense expansion of the
H-matrix's own factors (FP64 sums of at most 4096 terms on both sides).

Widths at and around the 16-column blocks and 64-column passes, leaves of 32
and 64, full and partial, factors in place and copied, the transposed plan,
and the mixed plan in its three modes.
"""
import numpy as np
import pytest

import hmx
import oracle as O
from test_gpu_pipeline import expand_gpu, to_dev

pytestmark = pytest.mark.gpu

WIDTHS = (2, 16, 17, 32, 33, 48, 64, 65)


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.fixture(scope="module", params=[(4096, 2, 32), (1111, 3, 32), (4096, 3, 64), (3001, 2, 64)],
                ids=["full-b32", "partial-b32", "full-b64", "partial-b64"])
def pipe(request, torch_cuda):
    n, d, b = request.param
    pp = hmx.Pipeline(n, d, b, 1e-6, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL,
                      points=to_dev(torch_cuda, O.generate_points(n, d, 31)), direct=True)
    pp.E = expand_gpu(pp.ctx, pp)
    yield pp
    hmx.lib().hmx_debug_set_wave_split(pp.H.handle, -1)


def both(pipe, f):
    out = []
    for split in (0, 1):
        assert hmx.lib().hmx_debug_set_wave_split(pipe.H.handle, split) == hmx.HMX_OK
        out.append(f().cpu().numpy())
    return out


@pytest.mark.parametrize("transpose", [False, True], ids=["forward", "transposed"])
@pytest.mark.parametrize("layout", [1, 2], ids=["in-place", "copied"])
def test_fp64(torch_cuda, pipe, layout, transpose):
    pipe.H.set_fp64_layout(layout)
    E = pipe.E.T if transpose else pipe.E
    for k in WIDTHS:
        X = O.generate_rhs(pipe.n, k, 3 + k)
        x = to_dev(torch_cuda, X.T)
        whole, split = both(pipe, lambda: pipe.matvec(x, transpose=transpose))
        assert np.array_equal(whole, split), k
        ref = E @ X
        assert np.linalg.norm(whole.T - ref) / np.linalg.norm(ref) < 1e-13, k


@pytest.mark.parametrize("mode", ["0", "1", "2"])
def test_mixed(torch_cuda, pipe, mode, monkeypatch):
    monkeypatch.setenv("HMX_MIXED_SPLIT", mode)
    pipe.make_mixed(3e-6)
    for k in WIDTHS:
        x = to_dev(torch_cuda, O.generate_rhs(pipe.n, k, 3 + k).T).float()
        whole, split = both(pipe, lambda: pipe.matvec_mixed(x))
        assert np.array_equal(whole, split), k
