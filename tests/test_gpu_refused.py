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
