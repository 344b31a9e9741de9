"""The library's held device memory: builds and products on two streams from
two threads at once, freeing and allocating blocks of the same sizes all the
time, give bit for bit what they give alone; and nothing is counted as live
once the handles are gone."""
import gc
import threading

import pytest

import hmx

pytestmark = pytest.mark.gpu

SIZES = [(1500, 2, 32), (4096, 3, 64), (2000, 2, 32)]


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def products(torch, ctx, stream, seed):
    out = []
    with torch.cuda.stream(stream):
        for n, d, b in SIZES:
            g = torch.Generator(device="cuda").manual_seed(seed + n)
            p = torch.rand(n * d, generator=g, device="cuda", dtype=torch.float64)
            x = torch.randn(5, n, generator=g, device="cuda", dtype=torch.float64)
            stream.synchronize()
            pipe = hmx.Pipeline(n, d, b, 1e-5, adm="maxDiam", max_rank_policy=hmx.MAXRANK_FULL, points=p, ctx=ctx,
                                direct=True)
            y1, y5 = torch.empty_like(x[0]), torch.empty_like(x)
            hmx.HMatrixVecMult(ctx, pipe.H, 1, x[0].contiguous(), y1)
            hmx.HMatrixVecMult(ctx, pipe.H, 5, x, y5)
            stream.synchronize()
            out += [y1.cpu(), y5.cpu()]
            del pipe
    return out


def test_two_threads_two_streams(torch_cuda):
    torch = torch_cuda
    ref = [products(torch, hmx.Context(s), s, seed) for seed, s in ((1, torch.cuda.Stream()), (2, torch.cuda.Stream()))]
    gc.collect()
    live0 = hmx.lib().hmx_debug_live_bytes()
    got, errors = {}, []

    def work(seed):
        try:
            s = torch.cuda.Stream()
            ctx = hmx.Context(s)
            got[seed] = [products(torch, ctx, s, seed) for _ in range(3)]
        except Exception as e:  # reported below
            errors.append(e)

    threads = [threading.Thread(target=work, args=(seed,)) for seed in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for seed in (1, 2):
        for out in got[seed]:
            assert all(torch.equal(a, b) for a, b in zip(out, ref[seed - 1]))
    gc.collect()
    assert hmx.lib().hmx_debug_live_bytes() == live0
