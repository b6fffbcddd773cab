"""Calls that a data error refuses write nothing, whatever route they take: the
outputs keep their old contents and the error arrives at sync."""
import pytest

from test_gpu_sweep import DT, _weights, rlq, say, torch

pytestmark = pytest.mark.gpu


def refused(ctx, index, column):
    with pytest.raises(rlq.QuantError) as e:
        ctx.sync()
    assert (e.value.name, e.value.index, e.value.b) == ("NonFiniteInput", index, column)


@pytest.mark.parametrize("t,cols,ncols", [(DT.Q4_K, 28672, 8), (DT.Q5_K, 28672, 8), (DT.Q4_K, 65536, 3),
                                          (DT.Q2_K, 65536, 3), (DT.Q3_K, 65536, 3), (DT.Q6_K, 4096, 2)],
                         ids=lambda v: v.name if isinstance(v, DT) else str(v))
def test_mul_mat_of_long_rows(t, cols, ncols):
    """Columns that do not fit one decode launch: an error in the last one holds
    back the first ones too."""
    say("refused mul_mat", t.name, cols, ncols)
    rows = 40
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, _weights(t, rows, cols, 3), rows, cols)
        x = torch.randn((1, 1, ncols, cols), generator=torch.Generator(device="cuda").manual_seed(4), device="cuda")
        y = torch.full((1, 1, ncols, rows), 7.0, device="cuda")
        x[..., -1, 300] = float("nan")
        ctx.mul_mat(W, x, y=y)
        refused(ctx, 300, ncols - 1)
        assert bool((y == 7.0).all())
        x[..., -1, 300] = 0.0
        ctx.mul_mat(W, x, y=y)
        ctx.sync()
        assert not bool((y == 7.0).any())
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("t,rows,cols,batch", [
    (DT.Q6_K, 300, 512, 12), (DT.Q8_0, 300, 96, 40), (DT.Q4_K, 300, 512, 12),  # int8 GEMM
    (DT.Q2_K, 64, 256, 262200),  # its folded flags
    (DT.Q3_K, 160016, 256, 9),  # keys of long rows
    (DT.Q4_K, 60000, 256, 96), (DT.Q4_K, 170000, 256, 130),  # f16 GEMM
], ids=lambda v: v.name if isinstance(v, DT) else str(v))
@pytest.mark.parametrize("noalloc", [False, True])
def test_argmax_of_many_columns(t, rows, cols, batch, noalloc):
    say("refused argmax", t.name, rows, cols, batch, "noalloc" if noalloc else "")
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, _weights(t, rows, cols, 5), rows, cols)
        x = torch.randn((batch, cols), generator=torch.Generator(device="cuda").manual_seed(6), device="cuda")
        y = torch.full((batch, rows), 7.0, device="cuda")
        best = torch.full((batch,), -5, dtype=torch.int32, device="cuda")
        call = (lambda: ctx.matmul_noalloc(W, x, y, best)) if noalloc else (lambda: ctx.matmul_argmax(W, x, y, best))
        x[-1, -1] = float("inf")
        call()
        refused(ctx, cols - 1, batch - 1)
        if not (noalloc and batch > 200000):  # (past the static scratch: passes of 8 columns)
            assert bool((y == 7.0).all()) and bool((best == -5).all())
        x[-1, -1] = 0.0
        call()
        ctx.sync()
        assert bool(((best >= 0) & (best < rows)).all())
        assert torch.equal(y.gather(1, best.long().view(-1, 1))[:, 0], y.amax(dim=1))
        W.close()
    finally:
        ctx.close()
