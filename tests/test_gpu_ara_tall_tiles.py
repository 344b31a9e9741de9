"""Tall tiles' column decisions and renormalisation with the column in registers
(4096, 8192 and 16384 rows) against the kernels that re-read it from memory:
the same sums in the same order, so ranks and factors are equal bit for bit --
the last columns of a tile are residuals that magnify any other rounding."""
import numpy as np
import pytest

import hmx
import oracle as O
from test_gpu_pipeline import to_dev

pytestmark = pytest.mark.gpu


def test_factors_are_equal_bit_for_bit(monkeypatch):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    n, b = 65536, 32
    pts = to_dev(torch, O.generate_points(n, 2, 17))
    ctx = hmx.Context()
    levels = {16384: 2, 8192: 3, 4096: 4}

    def factors():
        p = hmx.Pipeline(n, 2, b, 1e-5, adm="weak", max_rank_policy=hmx.MAXRANK_FULL, points=pts, ctx=ctx, direct=True)
        return {m: p.H.level(ctx, l) for m, l in levels.items()}

    regs = factors()
    monkeypatch.setenv("HMX_ARA_RELOAD", "1")
    reload = factors()
    for m in levels:
        (ra, Ua, Va), (rb, Ub, Vb) = regs[m], reload[m]
        assert Ua[0].shape[0] == m
        assert np.array_equal(ra, rb), m
        for t in range(len(ra)):
            assert np.array_equal(Ua[t], Ub[t]) and np.array_equal(Va[t], Vb[t]), (m, t)
