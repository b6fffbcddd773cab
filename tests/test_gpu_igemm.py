"""The int8 GEMM behind matmul of more than 8 columns, every weight format,
against the oracle: bitwise for Q8_0 and Q2_K (one f32 order), relative L2 <=
1e-5 per column for the others (exact block integers, another order of the
block terms; the bar of test_gpu_sweep).  The sizes sit at the edges of its
tiles (16-row layout tiles, 32-row wave tiles, 32-column tiles), at one block a
row, at K splits with fewer blocks than waves, at partial 256-value chunks and
odd block counts of Q8_0, and on both sides of its dispatch's tile counts (every
kernel with several chunks: test_gpu_igemm_exact).
"""
import numpy as np
import pytest

import oracle as O
from test_gpu_sweep import DT, EXACT_ALWAYS, REL_L2, TYPES, _weights, rel_l2, rlq, say, torch

pytestmark = pytest.mark.gpu

# (rows, 256-value blocks, columns).  The tile counts (32 rows x 32 columns) pass
# the dispatch's 160 (with 16 and more blocks: 16 waves), 512, 1024, 1700, 2048,
# 2700, 3000, 3500 and 4000.
SHAPES = ((1, 1, 33), (15, 1, 40), (17, 2, 65), (31, 3, 64), (33, 5, 97), (129, 9, 33), (47, 16, 65), (70, 35, 12),
          (2500, 9, 40), (9000, 2, 64), (18000, 1, 70), (22000, 1, 96), (16384, 2, 192), (30000, 1, 128), (32800, 1, 160))
Q8_0_COLS = (32, 96, 288, 544, 1120)


def cases():
    for t in TYPES:
        for rows, nb, batch in SHAPES:
            yield t, rows, nb * 256, batch
        yield t, 66000, 256, 31  # many tiles of one column tile each
        yield t, 131100, 256, 9
    for cols in Q8_0_COLS:
        yield DT.Q8_0, 70, cols, 47
    for t in (DT.Q3_K, DT.Q4_K, DT.Q5_K, DT.Q6_K):  # one column tile
        for batch in (9, 17, 32):
            yield t, 95, 2304, batch
    # two to eight columns on the GEMM
    for batch in (2, 3, 8):
        yield DT.Q6_K, 100, 4096, batch
    yield DT.Q6_K, 30, 512, 2
    for t in (DT.Q2_K, DT.Q3_K):
        yield t, 100, 2304, 5
        yield t, 17, 2048, 8
    yield DT.Q2_K, 4100, 8192, 3
    yield DT.Q8_0, 40, 32 * 331, 5
    yield DT.Q8_0, 4100, 4096, 8


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
        if batch > 8:  # (up to 8 columns an argmax takes the decode kernels)
            assert torch.equal(z, y[:batch])
        assert np.array_equal(best.cpu().numpy(), got.argmax(axis=1))
        got = z.cpu().numpy()
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


@pytest.mark.parametrize("rows,cols,batch", [(24500, 10272, 5), (24500, 10208, 5), (24600, 11264, 6), (24600, 14336, 5)])
def test_few_columns_of_long_rows(rows, cols, batch):
    """Q8_0 on both sides of the lines between the decode kernels and the GEMM:
    one f32 order, so bitwise the one-column products."""
    say("few columns", rows, cols, batch)
    gen = torch.Generator(device="cuda").manual_seed(cols)
    ctx = rlq.Context(0)
    try:
        w = ctx.quantize(DT.Q8_0, torch.randn((rows, cols), generator=gen, device="cuda")).reshape(-1)
        W = rlq.Weights(ctx, DT.Q8_0, w, rows, cols)
        x = torch.randn((batch, cols), generator=gen, device="cuda")
        y = ctx.matmul(W, x)
        ctx.sync()
        assert torch.equal(y, torch.cat([ctx.matmul(W, x[b:b + 1]) for b in range(batch)]))
        W.close()
    finally:
        ctx.close()


def test_flags_of_very_many_columns():
    """Past 8192 flags one launch folds them: slices of the result equal the
    slices' own products bit for bit, and the last column's error still
    suppresses every output."""
    say("igemm, 262176 columns")
    rows, cols, batch = 17, 256, 262176
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, DT.Q2_K, _weights(DT.Q2_K, rows, cols, 5), rows, cols)
        x = torch.randn((batch, cols), generator=torch.Generator(device="cuda").manual_seed(6), device="cuda")
        y = ctx.matmul(W, x)
        for i in (0, 131072, batch - 40):
            assert torch.equal(y[i:i + 40], ctx.matmul(W, x[i:i + 40]))
        ctx.sync()
        x[-1, -1] = float("nan")
        y.fill_(7.0)
        ctx.matmul(W, x, y)
        with pytest.raises(rlq.QuantError) as e:
            ctx.sync()
        assert (e.value.name, e.value.index, e.value.b) == ("NonFiniteInput", 255, batch - 1)
        assert bool((y == 7.0).all())
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("rows", [1, 63, 1025, 8192, 8200, 160000, 160016])
def test_argmax_of_many_columns(rows):
    """The first of equal maxima: every row occurs twice, and a zero column ties
    everywhere.  The lengths sit at the argmax kernels' strides (their lines:
    test_argmax_at_its_lines)."""
    say("argmax", rows)
    w = _weights(DT.Q4_K, (rows + 1) // 2, 256, rows).reshape(-1, 144)
    w = np.concatenate([w, w])[:rows].reshape(-1)
    x = np.random.default_rng(rows).standard_normal((10, 256)).astype(np.float32)
    x[4] = 0.0
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, DT.Q4_K, w, rows, 256)
        y, best = ctx.matmul_argmax(W, torch.from_numpy(x).cuda())
        z, same = torch.empty_like(y), torch.empty_like(best)
        ctx.matmul_noalloc(W, torch.from_numpy(x).cuda(), z, same)
        ctx.sync()
        assert np.array_equal(best.cpu().numpy(), y.cpu().numpy().argmax(axis=1))
        assert torch.equal(best, same) and torch.equal(y, z)
        W.close()
    finally:
        ctx.close()


# ---- several matrices -------------------------------------------------------------

def check(t, y, want):
    """y, want [products, rows]."""
    for i in range(len(want)):
        assert rel_l2(y[i], want[i]) <= REL_L2, i
    if t in EXACT_ALWAYS:
        assert np.array_equal(y.view(np.uint32), want.view(np.uint32))


def packed_rows(t, x):
    return np.concatenate([O.quantize(O.matvec_activation_dtype(int(t)), r) for r in x])


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("t", TYPES, ids=lambda t: DT(t).name)
def test_mul_mat_id_many_pairs(t, packed):
    """Enough pairs for the grouped products: experts without a token, tokens
    and slots without an expert, one expert with most tokens, and refusals by an
    id and by a column that no product uses."""
    rows, cols, experts, tokens, slots = 520, 2048, 6, 130, 2
    say("igemm ids", DT(t).name, "packed" if packed else "f32")
    w = _weights(t, experts * rows, cols, 7)
    rng = np.random.default_rng(8)
    ids = rng.integers(0, experts - 1, (tokens, slots)).astype(np.int32)  # the last expert unused
    ids[3:80, 0] = 2
    ids[5] = -1
    ids[9, 1] = -1
    x = rng.standard_normal((tokens, cols)).astype(np.float32)
    a = packed_rows(t, x) if packed else x
    xd = torch.from_numpy(a).cuda().reshape(tokens, 1, -1)
    at = O.matvec_activation_dtype(int(t)) if packed else O.F32
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, w, rows, cols, experts)
        y = ctx.mul_mat_id(W, xd, torch.from_numpy(ids).cuda(), x_dtype=at)
        ctx.sync()
        want = O.mul_mat_id(int(t), w, rows, cols, experts, at, a, 1, tokens, ids)
        check(t, y.cpu().numpy().reshape(-1, rows), np.asarray(want).reshape(-1, rows))
        z = torch.full((tokens, slots, rows), 7.0, device="cuda")
        bad = ids.copy()
        bad[100, 1], bad[101, 0] = experts, -2
        ctx.mul_mat_id(W, xd, torch.from_numpy(bad).cuda(), x_dtype=at, y=z)
        with pytest.raises(rlq.QuantError) as e:
            ctx.sync()
        assert (e.value.name, e.value.a) == ("Bounds", 201) and bool((z == 7.0).all())
        if not packed:
            xd[5, 0, 77] = float("nan")
            ctx.mul_mat_id(W, xd, torch.from_numpy(ids).cuda(), y=z)
            with pytest.raises(rlq.QuantError) as e:
                ctx.sync()
            assert (e.value.name, e.value.index, e.value.b) == ("NonFiniteInput", 77, 5) and bool((z == 7.0).all())
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("ncols", [2, 17, 33])
@pytest.mark.parametrize("t", TYPES, ids=lambda t: DT(t).name)
def test_mul_mat_broadcast_many_columns(t, ncols, packed):
    """Both broadcast directions: 2 matrices along n2 for 4 slices, along n3 for
    2, so that a matrix serves several runs of columns."""
    rows, cols, wn2, wn3, n2, n3 = 47, 768, 2, 1, 4, 2
    say("igemm broadcast", DT(t).name, ncols, "packed" if packed else "f32")
    w = _weights(t, wn2 * wn3 * rows, cols, 17)
    x = np.random.default_rng(18).standard_normal((n3 * n2 * ncols, cols)).astype(np.float32)
    a = packed_rows(t, x) if packed else x
    at = O.matvec_activation_dtype(int(t)) if packed else O.F32
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, w, rows, cols, wn2, wn3)
        xd = torch.from_numpy(a).cuda().reshape(n3, n2, ncols, -1)
        y = ctx.mul_mat(W, xd, x_dtype=at)
        ctx.sync()
        want = O.mul_mat(int(t), w, rows, cols, wn2, wn3, at, a, ncols, n2, n3)
        check(t, y.cpu().numpy().reshape(-1, rows), np.asarray(want).reshape(-1, rows))
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("rows,batch", [(28000, 10), (28001, 10), (28001, 256), (28001, 257), (160000, 257),
                                        (160001, 257)])
def test_argmax_at_its_lines(rows, batch):
    """One workgroup a column, or keys, on both sides of the lines between them;
    a zero column ties in every row."""
    say("argmax lines", rows, batch)
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, DT.Q8_0, _weights(DT.Q8_0, rows, 32, 5), rows, 32)
        x = torch.randn((batch, 32), generator=torch.Generator(device="cuda").manual_seed(6), device="cuda")
        x[1] = 0.0
        y, best = ctx.matmul_argmax(W, x)
        z, same = torch.empty_like(y), torch.empty_like(best)
        ctx.matmul_noalloc(W, x, z, same)
        ctx.sync()
        assert np.array_equal(best.cpu().numpy(), y.cpu().numpy().argmax(axis=1)) and int(best[1]) == 0
        assert torch.equal(best, same) and torch.equal(y, z)
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("rows,batch", [(16, 4194305), (160016, 65537)])
def test_argmax_of_very_many_columns(rows, batch):
    """More columns than one launch of the argmax kernels takes."""
    say("argmax", rows, "columns", batch)
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, DT.Q8_0, _weights(DT.Q8_0, rows, 32, 5), rows, 32)
        x = torch.randn((batch, 32), generator=torch.Generator(device="cuda").manual_seed(6), device="cuda")
        best = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
        y, _ = ctx.matmul_argmax(W, x, argmax=best)
        ctx.sync()
        assert bool(((best >= 0) & (best < rows)).all())
        assert torch.equal(y.gather(1, best.long().view(-1, 1))[:, 0], y.amax(dim=1))
        W.close()
    finally:
        ctx.close()
