"""Calls whose GEMM image does not fit the free device memory: they run the
decode kernels, which need far less, and give the GEMM's results."""
import pytest

from test_gpu_sweep import DT, REL_L2, _weights, rlq, say, torch

pytestmark = pytest.mark.gpu

ROWS, COLS, MATS = 16, 16384, 4
IMAGE = COLS // 256 * (9 * 1024 + 4)  # bytes per 32 columns


def calls():
    """name -> (matrices, image bytes, call(ctx, weights) -> y)"""
    gen = torch.Generator(device="cuda").manual_seed(8)
    many, groups, tokens, slots = 200000, 32766, 4000, 400

    def matmul():
        x = torch.randn((many, COLS), generator=gen, device="cuda")
        return 1, many // 32 * IMAGE, lambda ctx, w: ctx.matmul(w, x)

    def mul_mat():  # slices of two columns, each in a column tile of its own
        x = torch.randn((groups, 1, 2, COLS), generator=gen, device="cuda")
        return 1, groups * IMAGE, lambda ctx, w: ctx.mul_mat(w, x)

    def mul_mat_id():  # a column per (token, slot)
        x = torch.randn((tokens, 1, COLS), generator=gen, device="cuda")
        ids = torch.randint(0, MATS, (tokens, slots), generator=gen, device="cuda", dtype=torch.int32)
        return MATS, tokens * slots // 32 * IMAGE, lambda ctx, w: ctx.mul_mat_id(w, x, ids)

    return {"matmul": matmul, "mul_mat": mul_mat, "mul_mat_id": mul_mat_id}


@pytest.mark.parametrize("name", ["matmul", "mul_mat", "mul_mat_id"])
def test_image_past_the_free_memory(name):
    say("image past the free memory", name)
    mats, image, call = calls()[name]()
    data = _weights(DT.Q6_K, mats * ROWS, COLS, 7)

    def run():
        ctx = rlq.Context(0)
        try:
            W = rlq.Weights(ctx, DT.Q6_K, data, ROWS, COLS, mats)
            y = call(ctx, W)
            ctx.sync()
            W.close()
            return y
        finally:
            ctx.close()

    want = run()  # with the image
    torch.cuda.empty_cache()
    left = image // 2
    free = torch.cuda.mem_get_info()[0]
    if free < left:
        pytest.skip("less free memory than the call needs")
    fill = torch.empty(free - left, dtype=torch.uint8, device="cuda")
    try:
        say("free bytes", torch.cuda.mem_get_info()[0], "image", image)
        got = run()
    finally:
        del fill
        torch.cuda.empty_cache()
    error = (got - want).reshape(-1, ROWS).norm(dim=1)
    assert bool((error <= 2 * REL_L2 * want.reshape(-1, ROWS).norm(dim=1)).all())
