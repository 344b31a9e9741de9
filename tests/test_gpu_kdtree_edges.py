"""KD-tree sizes and inputs at the borders of the construction's kernels,
bitwise against the oracle: segments around the 2048 points that a workgroup
finishes in LDS, leaves of one point, radix passes of every count, chunks
around the radix kernels' 2048 points and the several-workgroup digit scan,
equal coordinates (grids, constant dimensions, few values) and infinities."""
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


@pytest.fixture(scope="module")
def ctx(torch_cuda):
    return hmx.Context()


def points(kind, n, d, seed):
    r = np.random.default_rng(seed)
    if kind == "uniform":
        return r.random(n * d)
    if kind == "grid":
        return r.integers(0, 16, n * d).astype(float) / 16
    if kind == "constant":  # one dimension of a single value, one of two
        p = r.random((d, n))
        p[0] = 0.5
        p[-1] = np.where(p[-1] < 0.5, -1.0, 1.0)
        return p.reshape(-1)
    if kind == "spread":  # magnitudes over 200 decades, both signs, zeros
        p = r.standard_normal(n * d) * 10.0 ** r.integers(-100, 100, n * d)
        p[r.integers(0, n * d, max(1, n // 10))] = 0.0
        return p
    p = r.random(n * d)
    p[r.integers(0, n * d, 4)] = np.inf
    p[r.integers(0, n * d, 4)] = -np.inf
    return p


def check(torch, ctx, p, n, d, b, div):
    tree = hmx.constructKDTree(ctx, n, d, b, to_dev(torch, p), divMethod=div)
    perm, off, lo, hi = tree.copy(ctx, n, d)
    if div == hmx.POWER_OF_TWO_ON_LEFT:
        ref = O.kdtree_pow2left(p, n, d, b)
    else:
        ref = O.kdtree(p, n, d, b)
    assert np.array_equal(perm, ref[0])
    assert np.array_equal(off, ref[1][:len(off)])
    levels = tree.info()[2]
    for level in range(levels):
        if div == hmx.POWER_OF_TWO_ON_LEFT:
            size = (1 << (int(n - 1).bit_length())) >> level
            cnt = -(-n // size)
        else:
            cnt = 1 << level
        a = (1 << level) - 1
        assert np.array_equal(lo[a:a + cnt], ref[2][a:a + cnt]), level
        assert np.array_equal(hi[a:a + cnt], ref[3][a:a + cnt]), level


@pytest.mark.parametrize("n,d,b", [(1, 2, 1), (2, 3, 1), (5, 1, 1), (64, 2, 64), (65, 2, 64), (2047, 3, 32),
                                   (2048, 2, 1), (2049, 2, 1), (2050, 3, 32), (4095, 1, 32), (4097, 3, 64),
                                   (40000, 3, 3000), (65535, 2, 64), (65537, 3, 32), (131073, 2, 32), (300001, 3, 64)])
def test_sizes(torch_cuda, ctx, n, d, b):
    check(torch_cuda, ctx, points("uniform", n, d, n), n, d, b, hmx.FULL_TREE)


@pytest.mark.parametrize("kind", ["grid", "constant", "spread", "infinite"])
@pytest.mark.parametrize("n,d,b", [(1500, 2, 8), (2100, 3, 16), (70000, 3, 32)])
def test_inputs(torch_cuda, ctx, kind, n, d, b):
    check(torch_cuda, ctx, points(kind, n, d, 3), n, d, b, hmx.FULL_TREE)


@pytest.mark.parametrize("n,d,b", [(1, 2, 4), (100, 2, 8), (2048, 3, 32), (2049, 2, 1), (3000, 3, 16), (5000, 2, 32),
                                   (70001, 3, 64)])
def test_power_of_two_on_left(torch_cuda, ctx, n, d, b):
    for kind in ("uniform", "grid"):
        check(torch_cuda, ctx, points(kind, n, d, 9), n, d, b, hmx.POWER_OF_TWO_ON_LEFT)
