"""The int8 GEMM behind matmul of more than 8 columns, every weight format,
against the oracle: bitwise for Q8_0 and Q2_K (one f32 order), relative L2 <=
1e-5 per column for the others (exact block integers, another order of the
block terms; the bar of test_gpu_sweep).  The sizes sit at the edges of its
tiles (16-row layout tiles, 32-row wave tiles, 32-column tiles), at one block a
row, at K splits with fewer blocks than waves, at partial 256-value chunks and
odd block counts of Q8_0, and on every workgroup shape of its dispatch.
"""
import numpy as np
import pytest

import oracle as O
from test_gpu_sweep import DT, EXACT_ALWAYS, REL_L2, TYPES, _weights, rel_l2, rlq, say, torch

pytestmark = pytest.mark.gpu

# (rows, 256-value blocks, columns): the row counts with 33 columns and more
# pass 512, 1100, 3000 and 4000 (32 x 32) tiles in turn
SHAPES = ((1, 1, 33), (15, 1, 40), (17, 2, 65), (31, 3, 64), (33, 5, 97), (129, 9, 33), (1000, 4, 36),
          (8200, 2, 64), (16500, 1, 130), (24600, 1, 128), (32800, 1, 160))
Q8_0_COLS = (32, 96, 288, 544, 1120)


def cases():
    for t in TYPES:
        for rows, nb, batch in SHAPES:
            yield t, rows, nb * 256, batch
    for cols in Q8_0_COLS:
        yield DT.Q8_0, 70, cols, 47
    for t in (DT.Q3_K, DT.Q4_K, DT.Q5_K, DT.Q6_K):  # one column tile
        for batch in (9, 17, 32):
            yield t, 95, 2304, batch


@pytest.mark.parametrize("t,rows,cols,batch", list(cases()), ids=lambda v: v.name if isinstance(v, DT) else str(v))
def test_many_columns(t, rows, cols, batch):
    say("igemm", DT(t).name, rows, cols, "columns", batch)
    w = _weights(t, rows, cols, rows + cols)
    x = np.random.default_rng(batch).standard_normal((batch, cols)).astype(np.float32)
    x[batch // 2] = 0.0  # a column whose blocks are all zero
    x[-1] = np.where(x[-1] < 0, np.float32(-3.0), np.float32(3.0))  # levels of +-127 throughout
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, w, rows, cols)
        y = torch.full((batch + 1, rows), 7.0, device="cuda")
        xd = torch.from_numpy(x).cuda()
        best = ctx.matmul_argmax(W, xd, y[:batch])[1]
        z = torch.empty((batch, rows), device="cuda")
        ctx.matmul_noalloc(W, xd, z)
        ctx.sync()
        got, want = y[:batch].cpu().numpy(), O.matmul(int(t), w, rows, cols, x, threads=16).reshape(batch, rows)
        assert bool((y[batch] == 7.0).all())
        assert torch.equal(z, y[:batch])
        assert np.array_equal(best.cpu().numpy(), got.argmax(axis=1))
        for b in range(batch):
            assert rel_l2(got[b], want[b]) <= REL_L2, b
        if t in EXACT_ALWAYS:
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        # the last column's last value not finite: its error, and nothing written
        xd[batch - 1, cols - 1] = float("inf")
        y.fill_(7.0)
        ctx.matmul(W, xd, y[:batch])
        with pytest.raises(rlq.QuantError) as e:
            ctx.sync()
        assert (e.value.name, e.value.index, e.value.b) == ("NonFiniteInput", cols - 1, batch - 1)
        assert bool((y == 7.0).all())
        W.close()
    finally:
        ctx.close()
