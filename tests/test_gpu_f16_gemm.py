"""The 128-column f16 GEMM of Q4_K (calls that fill its 256 row x 128 column
tiles; smaller ones run the int8 GEMM): ragged rows and columns, many column
tiles, the static scratch, the argmax after it and refused calls.  Each test
first asserts that the call runs that kernel.
"""
import numpy as np
import pytest
from torch.profiler import ProfilerActivity, profile

import oracle as O
from test_gpu_sweep import DT, REL_L2, _weights, rel_l2, rlq, say, torch

pytestmark = pytest.mark.gpu

# rows x values a row, columns: one round of the CUs, its last tiles partial
SHAPES = [(14330, 768, 500), (59999, 256, 97), (1790, 1024, 4100)]


def normal(seed, *shape):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def runs_the_gemm(ctx, call):
    call()  # (scratch allocated, kernels loaded)
    ctx.sync()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    ctx.sync()
    names = [e.key for e in p.key_averages()]
    return any("q4k_gemm_kernel" in n for n in names), names


@pytest.fixture(params=SHAPES, ids=lambda s: f"{s[0]}x{s[1]}-b{s[2]}")
def case(request):
    rows, cols, batch = request.param
    say("f16 GEMM", rows, cols, batch)
    ctx = rlq.Context(0)
    data = _weights(DT.Q4_K, rows, cols, rows)
    W = rlq.Weights(ctx, DT.Q4_K, data, rows, cols)
    yield ctx, W, data, rows, cols, batch, normal(batch, batch, cols)
    W.close()
    ctx.close()


def test_against_the_oracle(case):
    """Every column on sampled rows (the first and last tiles whole) against the
    oracle; every row of four columns against their one-column products, which
    are bitwise the oracle's."""
    ctx, W, data, rows, cols, batch, x = case
    y = torch.full((batch + 1, rows), 7.0, device="cuda")
    ran, names = runs_the_gemm(ctx, lambda: ctx.matmul(W, x, y[:batch]))
    assert ran, names
    sample = np.unique(np.r_[:40, 250:260, np.arange(0, rows, max(1, rows // 60)), rows - 40:rows])
    part = data.reshape(rows, -1)[sample].reshape(-1)
    want = O.matmul(O.Q4_K, part, sample.size, cols, x.cpu().numpy(), threads=16).reshape(batch, -1)
    got = y.cpu().numpy()
    assert (got[batch] == 7.0).all()
    for b in range(batch):
        assert rel_l2(got[b, sample], want[b]) <= REL_L2, b
    for b in (0, 31, 96, batch - 1):
        one = ctx.matmul(W, x[b:b + 1])[0].cpu().numpy()
        assert rel_l2(got[b], one) <= REL_L2, b


def test_argmax_and_static_scratch(case):
    ctx, W, _, rows, cols, batch, x = case
    y, best = ctx.matmul_argmax(W, x)
    z, same = torch.empty_like(y), torch.empty_like(best)
    ran, names = runs_the_gemm(ctx, lambda: ctx.matmul_noalloc(W, x, z, same))
    assert ran, names
    ctx.sync()
    assert torch.equal(y, z) and torch.equal(best, same)
    assert np.array_equal(best.cpu().numpy(), y.cpu().numpy().argmax(axis=1))


def test_refused(case):
    """A value of the last column not finite: its error, and nothing written."""
    ctx, W, _, rows, cols, batch, x = case
    y = torch.full((batch, rows), 7.0, device="cuda")
    best = torch.full((batch,), -5, dtype=torch.int32, device="cuda")
    x[-1, -1] = float("nan")
    for call in (lambda: ctx.matmul(W, x, y), lambda: ctx.matmul_argmax(W, x, y, best),
                 lambda: ctx.matmul_noalloc(W, x, y, best)):
        call()
        with pytest.raises(rlq.QuantError) as e:
            ctx.sync()
        assert (e.value.name, e.value.index, e.value.b) == ("NonFiniteInput", cols - 1, batch - 1)
        assert bool((y == 7.0).all()) and bool((best == -5).all())
