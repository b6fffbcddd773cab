"""The int8 GEMM's integers, bit for bit.  Weight blocks of random bytes with
super-scales of 1 (and minimum scales of 1) stand for whole numbers; activation
columns of whole numbers whose blocks peak at 127 are their own quantization, at
a scale of 1 or -1.  Every product, block sum and partial sum is then a whole
number, exact in f32 below 2^24 in whatever order it is added, so the result is
the 64-bit product itself: a lost carry between the weight planes, a stage read
too early or a K group left out shows in every format.

The sizes run every kernel of the dispatch with one chunk of 256 values and with
several, odd and even, so that stages, the K split and the refilled registers
are used again: by tiles of 32 rows x 32 columns (in brackets)
  up to 160, 16 or more chunks: 16 waves a tile; up to 512: 8; then 4 waves;
  [2304], [4617] columns in pairs: one column tile a wave (Q2_K, Q8_0), two with
  the K split (Q3_K, Q6_K) and without;  [4126] two column tiles;  [4097] one,
  which cannot pair.
"""
import numpy as np
import pytest

import oracle as O
from test_gpu_sweep import DT, TYPES, rlq, say, torch

pytestmark = pytest.mark.gpu

LIMIT = 2.0 ** 24
HALVES = {DT.Q8_0: (0,), DT.Q2_K: (80, 82), DT.Q3_K: (108,), DT.Q4_K: (0, 2), DT.Q5_K: (0, 2), DT.Q6_K: (208,)}


def blocks(t, rows, cols, seed, ends=False):
    """GGUF bytes [rows, row bytes], their whole numbers [rows, cols] and the
    part of them without the minimums, in 64 bits on the GPU.  ends: only the
    bytes whose fields are at the ends of their ranges."""
    rng = np.random.default_rng(seed)
    n, size = rows * (cols // O.BLOCK[int(t)]), O.TYPE_SIZE[int(t)]
    b = rng.choice(np.array([0, 255, 128, 127], np.uint8), (n, size)) if ends else \
        rng.integers(0, 256, (n, size), dtype=np.uint8)
    one = np.array([1.0], np.float16).view(np.uint8)
    for off in HALVES[t]:
        b[:, off:off + 2] = one
    values = []
    for minimum in (True, False):
        if not minimum and len(HALVES[t]) == 2:
            b = b.copy()
            b[:, HALVES[t][1]:HALVES[t][1] + 2] = 0
        if minimum:
            data = b.reshape(rows, -1)
        w = rlq.dequantize(t, b.reshape(-1), rows * cols)
        values.append(torch.from_numpy(w).cuda().to(torch.float64).view(rows, cols))
    return data, values[0], values[1]


def columns(t, batch, cols, most, seed):
    """[batch, cols] whole numbers in -most .. most, one of +-127 in each block."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randint(-most, most + 1, (batch, cols), generator=gen, device="cuda").to(torch.float32)
    peak = torch.randint(0, 2, (batch, cols // O.BLOCK[int(t)]), generator=gen, device="cuda") * 254.0 - 127.0
    x.view(batch, -1, O.BLOCK[int(t)])[:, :, seed % O.BLOCK[int(t)]] = peak
    return x


def fitting_columns(t, w, w0, batch, seed):
    """Columns as large as keep every partial sum, in any order, below 2^24."""
    most = 126
    while True:
        x = columns(t, batch, w.shape[1], most, seed)
        a = x.abs().to(torch.float64)
        if float((a @ w0.abs().t() + a @ (w0 - w).abs().t()).max()) < LIMIT:
            return x
        most //= 2
        assert most > 0


def exact(x, w):
    return (x.to(torch.float64) @ w.t()).to(torch.float32)


def shapes(t):
    for rows, nb, batch in ((47, 1, 9), (100, 17, 40), (95, 33, 20), (100, 3, 75), (4091, 3, 160), (4091, 6, 160)):
        yield rows, nb, batch
    for nb in (1, 2, 3, 4, 9):
        yield 8187, nb, 275
        yield 16390, nb, 275
    yield 7990, 3, 256  # [2000], [2008], [2176]: Q4_K's lines below and from four chunks
    yield 8010, 3, 256
    yield 8010, 1, 270
    yield 8010, 4, 256
    yield 66000, 3, 40
    yield 66000, 4, 64
    yield 131100, 3, 20


@pytest.mark.parametrize("t", TYPES, ids=lambda t: DT(t).name)
def test_products(t):
    ctx = rlq.Context(0)
    try:
        for rows, nb, batch in shapes(t):
            cols = nb * 256 - (96 if t == DT.Q8_0 else 0)  # (Q8_0: a partial chunk)
            say("exact", DT(t).name, rows, cols, batch)
            data, w, w0 = blocks(t, rows, cols, rows + nb)
            x = fitting_columns(t, w, w0, batch, nb)
            W = rlq.Weights(ctx, t, data.reshape(-1), rows, cols)
            y = ctx.matmul(W, x)
            ctx.sync()
            assert torch.equal(y, exact(x, w)), (rows, cols, batch)
            W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("rows,batch", [(300, 40), (16390, 275)])
@pytest.mark.parametrize("t", TYPES, ids=lambda t: DT(t).name)
def test_one_block_at_the_ends_of_its_ranges(t, rows, batch):
    """Levels and scales at the ends of their fields (Q6_K -128 * -32, Q5_K 63 *
    31) against columns of +-127 throughout, where the sum is below 2^24."""
    say("exact at the ends", DT(t).name, rows, batch)
    cols = O.BLOCK[int(t)]
    data, w, w0 = blocks(t, rows, cols, 3, ends=True)
    x = torch.randint(0, 2, (batch, cols), generator=torch.Generator(device="cuda").manual_seed(4),
                      device="cuda").to(torch.float32) * 254 - 127
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, data.reshape(-1), rows, cols)
        y = ctx.matmul(W, x)
        ctx.sync()
        fits = (exact(x, w).abs() < LIMIT) & (exact(x, w0).abs() < LIMIT) & (exact(x, w0 - w).abs() < LIMIT)
        assert float(fits.to(torch.float32).mean()) > 0.9
        assert torch.equal(y[fits], exact(x, w)[fits])
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("rows,nb,experts,tokens,counts", [
    (3187, 3, 3, 210, (129, 150, 131)), (3187, 4, 3, 210, (129, 150, 131)),  # pairs of tiles; K split of Q3_K, Q6_K
    (8187, 3, 3, 210, (129, 150, 131)), (8187, 4, 3, 210, (192, 64, 154)),
    (8187, 3, 6, 150, (1, 33, 64, 0, 150, 42))])  # single tiles
@pytest.mark.parametrize("t", TYPES, ids=lambda t: DT(t).name)
def test_dealt_products(t, rows, nb, experts, tokens, counts):
    """MUL_MAT_ID past the few-tile kernels: matrices with an empty second tile
    (129 products), without products, slots without a matrix and columns that no
    product uses."""
    cols = nb * 256 - (96 if t == DT.Q8_0 else 0)
    say("exact ids", DT(t).name, rows, cols, experts, tokens)
    data, w, w0 = blocks(t, experts * rows, cols, 7)
    x = fitting_columns(t, w, w0, tokens, 5)
    ids = np.full(tokens * 2, -1, np.int32)
    ids[2:2 + sum(counts)] = np.random.default_rng(6).permutation(np.repeat(np.arange(experts, dtype=np.int32), counts))
    ids = torch.from_numpy(ids.reshape(tokens, 2)).cuda()  # (token 0: no matrix)
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, data.reshape(-1), rows, cols, experts)
        y = ctx.mul_mat_id(W, x.view(tokens, 1, cols), ids)
        ctx.sync()
        w = w.view(experts, rows, cols)
        want = torch.zeros_like(y)
        for e in range(experts):
            token, slot = (ids == e).nonzero(as_tuple=True)
            want[token, slot] = exact(x[token], w[e])
        assert torch.equal(y, want)
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("rows,cols,tokens", [(4900, 832, 45), (4800, 832, 60), (4810, 832, 60)])
def test_dealt_q8_0_products_about_the_line(rows, cols, tokens):
    """Q8_0 products of 1694, 1800 and 1812 tiles (of which many are unused): the
    few-tile kernel to 1800, the staged one past it."""
    say("exact ids about the line", rows, cols, tokens)
    data, w, w0 = blocks(DT.Q8_0, 8 * rows, cols, 9)
    x = fitting_columns(DT.Q8_0, w, w0, tokens, 7)
    ids = torch.from_numpy(np.random.default_rng(8).integers(0, 8, (tokens, 1)).astype(np.int32)).cuda()
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, DT.Q8_0, data.reshape(-1), rows, cols, 8)
        y = ctx.mul_mat_id(W, x.view(tokens, 1, cols), ids)
        ctx.sync()
        want = torch.stack([exact(x[i:i + 1], w.view(8, rows, cols)[int(e)])[0] for i, e in enumerate(ids[:, 0].tolist())])
        assert torch.equal(y[:, 0], want)
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("t", TYPES, ids=lambda t: DT(t).name)
def test_dealt_products_of_several_columns(t):
    """MUL_MAT_ID whose slots take turns with a token's columns (slot s: column
    s % 3 of the token's)."""
    rows, experts, tokens, ncols, slots = 1500, 5, 70, 3, 6
    cols = 768 - (96 if t == DT.Q8_0 else 0)
    say("exact ids, several columns", DT(t).name)
    data, w, w0 = blocks(t, experts * rows, cols, 9)
    x = fitting_columns(t, w, w0, tokens * ncols, 7)
    ids = torch.from_numpy(np.random.default_rng(8).integers(-1, experts, (tokens, slots)).astype(np.int32)).cuda()
    ids[3] = -1  # (columns that no product uses)
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, data.reshape(-1), rows, cols, experts)
        y = ctx.mul_mat_id(W, x.view(tokens, ncols, cols), ids)
        ctx.sync()
        w, x = w.view(experts, rows, cols), x.view(tokens, ncols, cols)
        want = torch.zeros_like(y)
        for e in range(experts):
            token, slot = (ids == e).nonzero(as_tuple=True)
            want[token, slot] = exact(x[token, slot % ncols], w[e])
        assert torch.equal(y, want)
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("nb", [1, 3, 4])
@pytest.mark.parametrize("t", TYPES, ids=lambda t: DT(t).name)
def test_broadcast_products(t, nb, packed):
    """Two matrices for two slices of 70 columns each, past the few-tile kernels."""
    rows, ncols, cols = 16390, 70, nb * 256 - (96 if t == DT.Q8_0 else 0)
    say("exact broadcast", DT(t).name, rows, cols, "packed" if packed else "f32")
    data, w, w0 = blocks(t, 2 * rows, cols, 8)
    x = fitting_columns(t, w, w0, 4 * ncols, 6)
    at = rlq.matvec_activation_dtype(t)
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, data.reshape(-1), rows, cols, 2)
        xd = ctx.quantize(at, x).reshape(1, 4, ncols, -1) if packed else x.view(1, 4, ncols, cols)
        y = ctx.mul_mat(W, xd, at if packed else DT.F32)
        ctx.sync()
        want = torch.cat([exact(part, w[i * rows:(i + 1) * rows]) for i, part in enumerate(x.view(2, 2 * ncols, cols))])
        assert torch.equal(y.view(-1, rows), want)
        W.close()
    finally:
        ctx.close()
