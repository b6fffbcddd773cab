"""Products recorded in HIP graphs: every replay against the eager call of the
same inputs, with eager calls between the replays that grow the context's
scratch past what the graph was captured with.  The graph's own scratch must
outlive that growth: the freed memory would go to the tensors allocated here.
"""
import pytest

from test_gpu_sweep import DT, REL_L2, _weights, rel_l2, rlq, say, torch

pytestmark = pytest.mark.gpu


def normal(seed, *shape):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def capture(call):
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call()
    return graph


def grow(ctx, k):
    """An eager product of other weights whose image is larger each time, and
    tensors that take whatever memory it freed."""
    cols = 2048
    W = rlq.Weights(ctx, DT.Q6_K, _weights(DT.Q6_K, 64, cols, 3), 64, cols)
    ctx.matmul(W, normal(k, 2000 * (k + 1), cols))
    fill = [torch.full((n,), 1e30, device="cuda") for n in (1 << 10, 1 << 14, 1 << 18, 1 << 20)]
    ctx.sync()
    W.close()
    return fill


def products(ctx):
    """name -> (call(x, y), x, y): products whose captured launches use the
    context's scratch."""
    rows, cols = 300, 1024
    out = {}
    for t, batch in ((DT.Q4_K, 12), (DT.Q4_K, 8), (DT.Q5_K, 8), (DT.Q5_K, 20)):
        W = rlq.Weights(ctx, t, _weights(t, rows, cols, 9), rows, cols)
        out[f"{t.name}_{batch}"] = (lambda x, y, W=W: ctx.matmul(W, x, y), normal(2, batch, cols),
                                    torch.zeros((batch, rows), device="cuda"))
    for t in (DT.Q4_K, DT.Q6_K):
        W = rlq.Weights(ctx, t, _weights(t, 2 * rows, cols, 10), rows, cols, 2)
        out[f"{t.name}_mul_mat"] = (lambda x, y, W=W: ctx.mul_mat(W, x, y=y), normal(3, 1, 2, 3, cols),
                                    torch.zeros((1, 2, 3, rows), device="cuda"))
        ids = torch.tensor([[0, 1], [1, -1], [0, 0]], dtype=torch.int32, device="cuda")
        out[f"{t.name}_mul_mat_id"] = (lambda x, y, W=W, ids=ids: ctx.mul_mat_id(W, x, ids, y=y), normal(4, 3, 1, cols),
                                       torch.zeros((3, 2, rows), device="cuda"))
    return out


@pytest.mark.parametrize("name", ["Q4_K_12", "Q4_K_8", "Q5_K_8", "Q5_K_20", "Q4_K_mul_mat", "Q6_K_mul_mat",
                                  "Q4_K_mul_mat_id", "Q6_K_mul_mat_id"])
def test_recorded_scratch_outlives_growth(name):
    say("captured", name)
    ctx = rlq.Context(0)
    try:
        call, x, y = products(ctx)[name]
        call(x, y)  # the scratch that the capture needs
        graph = capture(lambda: call(x, y))
        want = torch.empty_like(y)
        for k in range(3):
            x.mul_(-1.5)
            call(x, want)
            ctx.sync()
            fill = grow(ctx, k)
            y.zero_()
            graph.replay()
            ctx.sync()
            # (Q5_K of 20 columns: decode passes recorded, a GEMM otherwise)
            for a, b in zip(y.reshape(-1, y.shape[-1]).cpu().numpy(), want.reshape(-1, y.shape[-1]).cpu().numpy()):
                assert rel_l2(a, b) <= 2 * REL_L2 if b.any() else not a.any(), k
            if name != "Q5_K_20":
                assert torch.equal(y, want), k
            assert all(bool((f == 1e30).all()) for f in fill), k
    finally:
        ctx.close()


@pytest.mark.parametrize("t", [DT.Q6_K, DT.Q8_0, DT.Q3_K, DT.Q2_K], ids=lambda t: t.name)
def test_many_columns_need_no_scratch(t):
    """A capture on a fresh context records decode passes: the replays equal the
    same columns in eager passes of 8 bit for bit, and the GEMM's result within
    the bars of both."""
    say("captured without scratch", t.name)
    rows, cols, batch = 18000, 1024, 12
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, _weights(t, rows, cols, 9), rows, cols)
        x, y = normal(2, batch, cols), torch.zeros((batch, rows), device="cuda")
        graph = capture(lambda: ctx.matmul(W, x, y))
        for k in range(3):
            x.mul_(-1.5)
            y.zero_()
            graph.replay()
            ctx.sync()
            # (of these shapes, up to 8 columns run the decode kernels)
            passes = torch.cat([ctx.matmul(W, x[:8]), ctx.matmul(W, x[8:])])
            whole = ctx.matmul(W, x)
            fill = grow(ctx, k)
            ctx.sync()
            assert torch.equal(y, passes), k
            for b in range(batch):
                assert rel_l2(y[b].cpu().numpy(), whole[b].cpu().numpy()) <= 2 * REL_L2, (k, b)
            del fill
        W.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("t,rows,eager", [(DT.Q6_K, 3000, (16, 4000, 100000)), (DT.Q4_K, 160016, (10, 300, 700))],
                         ids=["Q6_K", "Q4_K"])
def test_recorded_argmax_outlives_larger_calls(t, rows, eager):
    """Captured output heads of one column and of nine, replayed between argmax
    calls of ever more columns (Q4_K's of 160016 rows use one key a column)."""
    say("captured argmax", t.name, rows)
    cols = 256
    ctx = rlq.Context(0)
    try:
        W = rlq.Weights(ctx, t, _weights(t, rows, cols, 4), rows, cols)
        xs = [normal(5, 1, cols), normal(6, 9, cols)]
        ys = [torch.zeros((len(x), rows), device="cuda") for x in xs]
        bests = [torch.zeros(len(x), dtype=torch.int32, device="cuda") for x in xs]

        def heads():
            for x, y, best in zip(xs, ys, bests):
                ctx.matmul_argmax(W, x, y, best)

        heads()
        graph = capture(heads)
        for k, columns in enumerate(eager):
            for x in xs:
                x.mul_(-1.5)
            want = [ctx.matmul_argmax(W, x) for x in xs]
            ctx.matmul_argmax(W, normal(7 + k, columns, cols))
            ctx.sync()
            fill = [torch.full((n,), 1e30, device="cuda") for n in (1 << 10, 1 << 12, 1 << 16)]
            for best in bests:
                best.fill_(-1)
            graph.replay()
            ctx.sync()
            for y, best, (z, index) in zip(ys, bests, want):
                assert torch.equal(best, y.argmax(dim=1).to(torch.int32)), k
                assert torch.equal(index, z.argmax(dim=1).to(torch.int32)), k
                assert all(rel_l2(a, b) <= 2 * REL_L2 for a, b in zip(y.cpu().numpy(), z.cpu().numpy())), k
            assert all(bool((f == 1e30).all()) for f in fill), k
        W.close()
    finally:
        ctx.close()
