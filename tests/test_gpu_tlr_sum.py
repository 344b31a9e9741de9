"""Upper levels compressed from the sum of a tile's leaf pairs, at leaf sizes
on either side of the sampler's row groups (16, 32 and 64 rows) and at tile
heights from two leaves on, against the oracle's H-matrix of the same random
numbers.

Bars: at most one rank differs by 1 per level (a column whose residual sits on
the tolerance may fall either way when the sums are ordered differently); the
error against the dense matrix is at most 1.5 times the oracle's.
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


@pytest.mark.parametrize("n,b", [(128, 16), (512, 16), (500, 32), (512, 64), (2000, 64)])
def test_levels_from_leaf_sums(torch_cuda, n, b):
    p = O.generate_points(n, 2, 11)
    ctx = hmx.Context()
    pipe = hmx.Pipeline(n, 2, b, 1e-6, adm="weak", max_rank_policy=hmx.MAXRANK_FULL, points=to_dev(torch_cuda, p),
                        ctx=ctx, seed=1234)
    ref = O.OracleHMatrix(p, n, 2, b, adm="weak", tol=1e-6, max_rank_policy=hmx.MAXRANK_FULL, seed=1234)
    for l in range(1, pipe.H.num_levels):
        d = np.abs(pipe.H.level(ctx, l)[0].astype(int) - ref.level(l)[0].astype(int))
        print(f"n={n} b={b} level {l}: {len(d)} tiles, rank differences {d.sum()}")
        assert d.sum() <= 1, l
    K = O.dense_matrix(p, n, 2, ref.perm, ref.ell)
    eg = np.linalg.norm(expand_gpu(ctx, pipe) - K) / np.linalg.norm(K)
    eo = np.linalg.norm(ref.expand() - K) / np.linalg.norm(K)
    assert eg <= 1.5 * eo + 1e-9
