"""Extended row tiles of the 128-row LDS-DMA kernels (tile policies 5 and 14):
the last tile of a group also takes up to 32 rows past its 128. Groups of
exactly the sizes at the rule's edges (one tile up to 160 rows, two up to 288)
against the CPU oracle, on both combine paths, in overwrite and accumulate
mode, with K and column tails, and pre-packed weights bit for bit against the
API layout. Tolerances as tests/test_gpu_moe.py."""
import ctypes

import numpy as np
import pytest

import candle_moe
import oracle as O
from helpers import RTOL, assert_close, from_dev, moe_inputs, to_dev

pytestmark = pytest.mark.gpu

# rows per expert: one row, a full tile, extensions of 1, 31 and 32 rows, one
# row too many, two tiles with and without extension
SIZES = [1, 128, 129, 159, 160, 161, 256, 257, 288, 289, 0]


def _routing(k):
    """Indices [T, k] (a token's experts distinct) giving expert e SIZES[e] of the first slots."""
    rng = np.random.RandomState(7)
    first = np.repeat(np.arange(len(SIZES)), SIZES)
    rng.shuffle(first)
    T, E = len(first), len(SIZES) + k - 1
    idx = np.empty((T, k), dtype=np.uint32)
    idx[:, 0] = first
    for j in range(1, k):  # further slots: experts of their own (T rows each)
        idx[:, j] = len(SIZES) + j - 1
    w = rng.uniform(0.1, 1.0, size=(T, k)).astype(np.float32)
    return T, E, idx, w


@pytest.mark.parametrize("tile", [5, 14])
@pytest.mark.parametrize("mt,dt,H,I,k", [(O.QWEN3, O.BF16, 200, 136, 1), (O.QWEN3, O.F16, 264, 192, 2),
                                         (O.NOMIC, O.BF16, 136, 328, 2), (O.NOMIC, O.F16, 72, 256, 1)])
def test_extended_tiles(tile, mt, dt, H, I, k):
    import torch

    T, E, idx, w = _routing(k)
    act = O.SILU if mt == O.QWEN3 else O.GELU
    x, G, U, D, _, _ = moe_inputs(T, H, I, E, 1, dt, 500 + tile + H, mt)
    want = O.fused_moe(x, G, U, D, w, idx, E=E, k=k, act=act, moe_type=mt, dtype=dt, mode=O.MODE_F32ACC)
    tx, tg, tu, tw, ti = to_dev(x, dt), to_dev(G, dt), to_dev(U, dt), to_dev(w), to_dev(idx)
    td = to_dev(D, dt) if D is not None else None
    moe = candle_moe.FusedMoE.new(E, k, candle_moe.Activation(act))
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None  # noqa: E731
    try:
        candle_moe.set_tile_policy(tile)
        for combine in (candle_moe.COMBINE_PAIRS, candle_moe.COMBINE_EXPERT_SETS):
            candle_moe.set_combine_policy(combine)
            got = moe.forward(tx, tg, tu, td, tw, ti, mt)  # overwrite
            acc = torch.ones_like(got)
            candle_moe.check(candle_moe.lib().candle_moe_fused_moe_status(
                p(tx), p(tg), p(tu), p(td), p(tw), p(ti), p(acc), T, H, I, E, k, act, mt, dt,
                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
            torch.cuda.synchronize()
            what = f"tile {tile} combine {combine}"
            assert_close(from_dev(got), want, RTOL[dt], what)
            assert_close(from_dev(acc), want + 1.0, RTOL[dt], what + " accumulate")
        candle_moe.set_combine_policy(candle_moe.COMBINE_PAIRS)
        got = moe.forward(tx, tg, tu, td, tw, ti, mt)
        packed = torch.zeros_like(got)
        candle_moe.fused_moe_packed(tx, candle_moe.pack_weights(tg), candle_moe.pack_weights(tu) if td is not None else tu,
                                    candle_moe.pack_weights(td) if td is not None else None, tw, ti, packed, E, k, act, mt)
        torch.cuda.synchronize()
        assert torch.equal(got, packed)
    finally:
        candle_moe.set_tile_policy(0)
        candle_moe.set_combine_policy(candle_moe.COMBINE_AUTO)
