"""The weight encoders' searches at their edges, byte for byte the oracle's: flat,
zero and negative-zero blocks, one-signed blocks, sub-blocks of zeros or of one
outlier, values whose super-scale is subnormal, two-valued blocks.
"""
import numpy as np
import pytest

import oracle as O
from rlq_loader import load

rlq = load()
torch = rlq.torch
DT = rlq.DType

pytestmark = pytest.mark.gpu


def rows(cols):
    rng = np.random.default_rng(3)
    x = (rng.standard_normal((14, cols)) * 0.02).astype(np.float32)
    x[0] = 0.0
    x[1] = 1.5
    x[2] = -0.25
    x[3, :64] = 0.0
    x[4] *= np.float32(1e-7)
    x[5] = np.abs(x[5])
    x[6] = -np.abs(x[6])
    x[7] *= np.float32(1e4)
    x[8, ::2] = 0.0
    x[9] = np.round(x[9] * 100)
    x[10, 5] = 30.0
    x[11] = -0.0
    x[12] = np.sign(x[12]) * np.float32(0.5)
    return x


@pytest.mark.parametrize("t", [DT.Q2_K, DT.Q3_K, DT.Q4_K, DT.Q5_K, DT.Q6_K], ids=lambda t: t.name)
@pytest.mark.parametrize("cols", [256, 768])
def test_edges(t, cols):
    print("[case] encode edges", t.name, cols, flush=True)
    x = rows(cols)
    ctx = rlq.Context(0)
    try:
        got = ctx.quantize(t, torch.from_numpy(x).cuda())
        ctx.sync()
        assert np.array_equal(got.cpu().numpy(), np.concatenate([O.quantize(int(t), r) for r in x]))
    finally:
        ctx.close()
