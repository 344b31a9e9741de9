"""One right-hand side through the streaming kernels against the dense
expansion of the H-matrix's own factors: columns inside one work item and
columns in several chunks, leaves with fewer tiles than a workgroup has parts,
full and partial leaves, both directions; nothing is written past the vector.

Bar: 1e-13 of the norm, as for the other products (FP64 sums of at most 9000
terms on both sides).
"""
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


@pytest.mark.parametrize("n,d,b,adm", [(65, 2, 32, "maxDiam"), (128, 2, 64, "weak"), (1000, 2, 32, "maxDiam"),
                                       (4096, 3, 64, "maxDiam"), (8192, 2, 32, "weak"), (9000, 2, 64, "weak")])
def test_one_right_hand_side(torch_cuda, n, d, b, adm):
    torch = torch_cuda
    pp = hmx.Pipeline(n, d, b, 1e-6, adm=adm, max_rank_policy=hmx.MAXRANK_FULL,
                      points=to_dev(torch, O.generate_points(n, d, 31)), direct=True)
    E = torch.from_numpy(expand_gpu(pp.ctx, pp)).cuda()
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
    for t in (False, True):
        out = torch.full((n + 64,), float("nan"), device="cuda", dtype=torch.float64)
        y = pp.matvec(x, out[:n], transpose=t)
        ref = torch.mv(E.t() if t else E, x)
        rel = float(torch.linalg.norm(y - ref) / torch.linalg.norm(ref))
        print(f"n={n} d={d} b={b} {adm} transpose={t}: rel {rel:.2e}")
        assert rel < 1e-13
        assert bool(torch.isnan(out[n:]).all())
