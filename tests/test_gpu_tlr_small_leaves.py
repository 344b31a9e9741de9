"""Upper levels compressed from leaf pairs of 8 rows, half of the sampler's
16-row group masked, from two leaves a side on and with partial leaves, against
the oracle's H-matrix of the same random numbers.

Bars as for the other leaf sizes: at most one rank differs by 1 per level, the
error against the dense matrix is at most 1.5 times the oracle's.
"""
import numpy as np
import pytest

import hmx
import oracle as O
from test_gpu_pipeline import expand_gpu, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32, 61, 64, 256, 500])
def test_levels_from_leaf_sums_of_8_rows(n):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    b = 8
    p = O.generate_points(n, 2, 11)
    ctx = hmx.Context()
    pipe = hmx.Pipeline(n, 2, b, 1e-6, adm="weak", max_rank_policy=hmx.MAXRANK_FULL, points=to_dev(torch, p), ctx=ctx,
                        seed=1234)
    ref = O.OracleHMatrix(p, n, 2, b, adm="weak", tol=1e-6, max_rank_policy=hmx.MAXRANK_FULL, seed=1234)
    for l in range(1, pipe.H.num_levels):
        d = np.abs(pipe.H.level(ctx, l)[0].astype(int) - ref.level(l)[0].astype(int))
        assert d.sum() <= 1, l
    K = O.dense_matrix(p, n, 2, ref.perm, ref.ell)
    eg = np.linalg.norm(expand_gpu(ctx, pipe) - K) / np.linalg.norm(K)
    eo = np.linalg.norm(ref.expand() - K) / np.linalg.norm(K)
    assert eg <= 1.5 * eo + 1e-9
