"""Factor gradients of every tile against the same outer products in torch.

dU_t = dY[rows] (V_t^T X[cols])^T and dV_t = X[cols] (U_t^T dY[rows])^T from
the library's own factors, all levels: tiles taken by one wave (below 512
rows) and by a workgroup (512 and more), ranks around the 16- and 32-column
blocks of an item, right-hand sides around the 16-column blocks and the
64-column passes of the kernel, partial leaves, and vectors that start 8
bytes past a 16-byte boundary.

Bar: both sides sum m + k products in FP64, so they differ by at most
2 (m + k) 2^-53 of the sums of absolute values; with m <= 1024, k <= 130 and
random signs (the sums are sqrt(m) below the sums of absolute values) 1e-12
of the gradient's norm.
"""
import ctypes

import numpy as np
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


@pytest.fixture(scope="module", params=[(2048, 2, 32, "weak"), (4096, 2, 64, "maxDiam"), (1500, 3, 64, "weak")],
                ids=["full-2d-b32", "full-2d-b64", "partial-3d-b64"])
def pipe(request, torch_cuda):
    n, d, b, adm = request.param
    p = O.generate_points(n, d, 17)
    return hmx.Pipeline(n, d, b, 1e-6, adm=adm, max_rank_policy=hmx.MAXRANK_FULL, points=to_dev(torch_cuda, p),
                        direct=True)


def vectors(torch, k, n, seed, skew):
    g = torch.Generator(device="cuda").manual_seed(seed)
    buf = torch.randn(k * n + 2, generator=g, device="cuda", dtype=torch.float64)
    return buf[skew:skew + k * n].view(k, n)


@pytest.mark.parametrize("k,skew", [(1, 0), (15, 1), (16, 0), (17, 0), (33, 0), (64, 1), (65, 0), (130, 0)])
def test_gradients_of_every_tile(torch_cuda, pipe, k, skew):
    torch = torch_cuda
    n, b, S, L = pipe.n, pipe.b, pipe.tree.info()[0], pipe.H.num_levels
    X, W = vectors(torch, k, n, k, skew), vectors(torch, k, n, 1000 + k, skew)
    levels = [l for l in range(1, L) if pipe.H.level_info(l)["rankSum"]]
    fac = {l: pipe.H.level_device(pipe.ctx, l) for l in levels}
    dU = {l: torch.full_like(fac[l][0], float("nan")) for l in levels}
    dV = {l: torch.full_like(fac[l][1], float("nan")) for l in levels}
    table = lambda d: (ctypes.c_void_p * (L - 1))(*[d[l].data_ptr() if l in d else 0 for l in range(1, L)])
    hmx._check(hmx.lib().hmx_hmatvec_grad_factors(pipe.ctx.handle, pipe.H.handle, k, hmx._ptr(X), hmx._ptr(W),
                                                  table(dU), table(dV)), pipe.ctx)
    offs = pipe.tree.copy(pipe.ctx, n, pipe.d)[1]
    pos = np.concatenate([q * b + np.arange(offs[q + 1] - offs[q]) for q in range(S)])
    pad = lambda x: torch.zeros(k, S * b, device="cuda", dtype=torch.float64).index_copy_(
        1, torch.from_numpy(pos).cuda(), x.contiguous())
    Xp, Wp = pad(X), pad(W)
    for l in levels:
        m = (1 << (L - 1 - l)) * b
        ranks, tiles = pipe.H.level_ranks(pipe.ctx, l), pipe.structure.tiles(l)
        U, V = (f.view(-1, m) for f in fac[l])
        c0 = 0
        refU, refV = torch.empty_like(U), torch.empty_like(V)
        for t, r in enumerate(ranks):
            u, v = O._mo_to_xy(int(tiles[t]))
            x, w = Xp[:, u * m:(u + 1) * m], Wp[:, v * m:(v + 1) * m]
            refU[c0:c0 + r] = (V[c0:c0 + r] @ x.T) @ w
            refV[c0:c0 + r] = (U[c0:c0 + r] @ w.T) @ x
            c0 += r
        for got, ref in ((dU[l], refU), (dV[l], refV)):
            err = float(torch.linalg.norm(got.view(-1, m) - ref) / torch.linalg.norm(ref))
            assert err <= 1e-12, (l, m, k, err)
