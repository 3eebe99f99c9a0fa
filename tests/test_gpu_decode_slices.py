"""Decode kernels whose gate/up GEMM has few, long 64-column blocks: K slices and
a finishing launch by default. Both sides of the line (block length H = 4096,
number of blocks) with K and column tails, API layout and pre-packed weights,
against the CPU oracle. Tolerances as tests/test_gpu_moe.py."""
import numpy as np
import pytest
import torch

import candle_moe
import oracle as O
from helpers import RTOL, assert_close, from_dev, moe_inputs, to_dev
from test_gpu_moe import check_case

pytestmark = pytest.mark.gpu

CASES = [  # T, H, I, E, k: blocks = min(T k, E) * ceil(I / 64)
    (1, 4096, 136, 4, 2), (1, 4104, 136, 4, 1), (2, 4088, 136, 4, 2),   # 6 and 3 blocks; too short: one slice
    (2, 4096, 264, 16, 6), (2, 4096, 328, 16, 6), (3, 4200, 8, 4, 2),   # 60, 72 blocks; blocks of 8 columns
]


@pytest.mark.parametrize("T,H,I,E,k", CASES)
@pytest.mark.parametrize("dt", [O.BF16, O.F16])
def test_api_layout(T, H, I, E, k, dt):
    assert candle_moe.fused_moe_kernel(T, H, I, E, k, dt) == candle_moe.TILE_DEC_GEMV
    check_case(T, H, I, E, k, dt, O.QWEN3, act=O.SILU, seed=900 + T + I)


@pytest.mark.parametrize("T,H,I,E,k", [(1, 4096, 136, 4, 2), (2, 4104, 264, 16, 6), (2, 4096, 328, 16, 6)])
def test_packed(T, H, I, E, k):  # 6, 60 and 72 blocks (the line is at 64); bit for bit the API layout
    dt = O.BF16
    x, G, U, D, rw, ri = moe_inputs(T, H, I, E, k, dt, 930 + T + I, O.QWEN3)
    want = O.fused_moe(x, G, U, D, rw, ri, E=E, k=k, act=O.SILU, moe_type=O.QWEN3, dtype=dt, mode=O.MODE_F32ACC)
    tx, trw, tri = to_dev(x, dt), to_dev(rw), to_dev(ri)
    out = torch.zeros_like(tx)
    packed = [candle_moe.pack_weights(to_dev(w, dt)) for w in (G, U, D)]
    candle_moe.fused_moe_packed(tx, *packed, trw, tri, out, E, k)
    torch.cuda.synchronize()
    assert_close(from_dev(out).astype(np.float64), want, RTOL[dt], f"packed T={T} I={I}")
    api = candle_moe.FusedMoE.new(E, k, candle_moe.Activation.Silu).forward(
        tx, to_dev(G, dt), to_dev(U, dt), to_dev(D, dt), trw, tri, 0)
    assert torch.equal(api, out)
