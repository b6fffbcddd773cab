"""Calls whose GEMM launches would pass 2^32 threads (HIP then runs a part of the
grid and reports nothing): they take the decode kernels and give the same bits
as calls of their parts."""
import pytest

from test_gpu_sweep import DT, _weights, rlq, say, torch

pytestmark = pytest.mark.gpu


def normal(seed, *shape):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def test_mul_mat_of_many_groups():
    """One matrix for 32766 slices of two columns, each in a column tile of its own."""
    rows, cols, slices = 65537, 32, 32766
    say("mul_mat", rows, cols, slices)
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, DT.Q8_0, _weights(DT.Q8_0, rows, cols, 1), rows, cols)
        x = normal(2, slices, 1, 2, cols)
        y = torch.full((slices, 1, 2, rows), 7.0, device="cuda")
        ctx.mul_mat(W, x, y=y)
        for i in (0, 1000, 20000, slices - 500):
            same = torch.equal(y[i:i + 500].view(1000, rows), ctx.matmul(W, x[i:i + 500].view(1000, cols)))
            assert same, i
        ctx.sync()
        W.close()
    finally:
        ctx.close()


def test_mul_mat_id_of_many_products():
    """An image of more than 2^23 (column tile, chunk) records."""
    rows, cols, tokens, slots = 16, 8448, 65535, 128
    say("mul_mat_id", rows, cols, tokens, slots)
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, DT.Q8_0, _weights(DT.Q8_0, 2 * rows, cols, 1), rows, cols, 2)
        x = normal(3, tokens, 1, cols)
        ids = torch.randint(0, 2, (tokens, slots), generator=torch.Generator(device="cuda").manual_seed(4), device="cuda",
                            dtype=torch.int32)
        y = torch.full((tokens, slots, rows), 7.0, device="cuda")
        ctx.mul_mat_id(W, x, ids, y=y)
        for i in (0, 30000, tokens - 300):
            same = torch.equal(y[i:i + 300], ctx.mul_mat_id(W, x[i:i + 300].contiguous(), ids[i:i + 300].contiguous()))
            assert same, i
        ctx.sync()
        W.close()
    finally:
        ctx.close()
