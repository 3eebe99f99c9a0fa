"""f32 MoE on the bf16 matrix cores (three-part split): accuracy at tile and
K-step edges, and inputs the split cannot hold.

Error bound of the accuracy cases (2-norm, relative to the 64-bit result).
Every product keeps all but 2^-26 of itself; the large part products are
accumulated in f32, one rounding per 16 k: at K <= 512 per GEMM at most 32
roundings of 2^-24 each in a worst case that random signs do not reach, twice
(two GEMMs), plus a few ulp of the activation and the final roundings:
2 * 32 * 2^-24 + 4 * 2^-23 = 4.3e-6. A dropped part product of relative size
2^-16 or a bf16-rounded operand would show at 1e-5 and above.
"""
import numpy as np
import pytest

import candle_moe
import oracle as O
from helpers import moe_inputs, to_dev, from_dev

pytestmark = pytest.mark.gpu

REL = 4.3e-6


def _forward(x, G, U, D, rw, ri, E, k, act, mt, tile):
    import torch

    try:
        candle_moe.set_tile_policy(tile)
        moe = candle_moe.FusedMoE.new(E, k, candle_moe.Activation(act))
        out = moe.forward(to_dev(x), to_dev(G), to_dev(U), to_dev(D) if D is not None else None, to_dev(rw),
                          to_dev(ri), mt)
        torch.cuda.synchronize()
        return from_dev(out)
    finally:
        candle_moe.set_tile_policy(0)


# tile 0: the default (decode kernels up to 256 pairs), 15 / 16: 32- and
# 128-row tiles; row counts around 16, 32, 64 and 128 per expert, columns
# around 64 and 128, K around the 32- and 64-deep steps, single-expert runs
@pytest.mark.parametrize("tile,T,H,I,E,k,mt", [
    (0, 1, 8, 8, 1, 1, 0), (0, 1, 768, 96, 8, 2, 1), (0, 16, 104, 200, 1, 1, 0), (0, 17, 512, 136, 3, 2, 1),
    (0, 33, 72, 264, 2, 2, 0), (0, 128, 128, 64, 8, 2, 1), (18, 70, 256, 72, 2, 1, 0), (18, 70, 264, 56, 2, 1, 1),
    (15, 31, 60, 132, 1, 1, 0), (15, 65, 68, 124, 2, 1, 1), (15, 32, 512, 64, 1, 1, 0), (15, 9, 4, 4, 2, 2, 1),
    (16, 127, 100, 68, 1, 1, 0), (16, 129, 132, 260, 1, 1, 1), (16, 65, 36, 128, 1, 1, 0), (16, 3, 512, 192, 2, 1, 1),
])
def test_f32_split_accuracy(tile, T, H, I, E, k, mt):
    act = O.SILU if mt == 0 else O.GELU
    x, G, U, D, rw, ri = moe_inputs(T, H, I, E, k, O.F32, 900 + T + H, mt)
    got = _forward(x, G, U, D, rw, ri, E, k, act, mt, tile).astype(np.float64)
    want = O.fused_moe(x, G, U, D, rw, ri, E=E, k=k, act=act, moe_type=mt, dtype=O.F32, mode=O.MODE_EXACT)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= REL, err


@pytest.mark.parametrize("tile", [0, 15, 16])
@pytest.mark.parametrize("mt", [O.QWEN3, O.NOMIC])
def test_f32_split_non_finite_and_extreme_inputs(tile, mt):
    # an infinity, a NaN, a value whose bf16 part would round to infinity and
    # values whose low parts would be subnormal unscaled: what f32 FMAs give. (ReLU: an
    # infinite pre-activation stays infinite or becomes zero.)
    T, H, I, E, k = 40, 64, 72, 2, 1
    x, G, U, D, rw, ri = moe_inputs(T, H, I, E, k, O.F32, 950, mt)
    x[3, 5] = np.inf
    x[4, 7] = -np.inf
    x[9, 0] = np.nan
    x[10, 1] = np.float32(3.4e38)
    x[11, :] *= np.float32(1e-34)
    x[12, :] = 0.0
    G[0, 6, 3] = np.float32(0.5)  # parts m and l are zero: inf * 0 must not appear
    got = _forward(x, G, U, D, rw, ri, E, k, O.RELU, mt, tile)
    want = O.fused_moe(x, G, U, D, rw, ri, E=E, k=k, act=O.RELU, moe_type=mt, dtype=O.F32, mode=O.MODE_F32ACC)
    for t in range(T):
        g, w = got[t].astype(np.float64), np.asarray(want[t], dtype=np.float64)
        if t in (3, 4, 9):
            assert np.array_equal(np.isnan(g), np.isnan(w)), t
            fin = ~np.isnan(w)
            assert np.array_equal(g[fin], w[fin]) or np.allclose(g[fin], w[fin], rtol=1e-4), t
        else:
            assert np.isfinite(w).all() == np.isfinite(g).all(), t
            if np.isfinite(w).all():
                assert np.linalg.norm(g - w) <= 1e-5 * np.linalg.norm(w) + 1e-44, t


@pytest.mark.parametrize("tile", [0, 15, 16])
@pytest.mark.parametrize("mt,tiny", [(O.NOMIC, "x"), (O.NOMIC, "gate"), (O.NOMIC, "up"), (O.QWEN3, "gate"), (O.QWEN3, "down")])
@pytest.mark.parametrize("scale", [1e-36, 1e-38, 1e-41])
def test_f32_split_tiny_operands(tile, mt, tiny, scale):
    """One operand tiny, subnormal ones included, the others such that every sum
    stays in f32's normal range: the parts still hold every bit, so the bound is
    that of ordinary values. (Unscaled parts lost the bits below 2^-133: 2.6e-5
    at 1e-36, 2.6e-3 at 1e-38.)"""
    T, H, I, E, k = 40, 256, 192, 2, 1
    x, G, U, D, rw, ri = moe_inputs(T, H, I, E, k, O.F32, 970, mt, wstd=1.0)
    ops = {"x": x, "gate": G, "up": U, "down": D}
    for name, t in ops.items():
        if t is not None:
            t *= np.float32(scale if name == tiny else 100.0)
    G *= np.float32(100.0 if tiny != "gate" else 1.0)
    got = _forward(x, G, U, D, rw, ri, E, k, O.RELU, mt, tile).astype(np.float64)
    want = O.fused_moe(x, G, U, D, rw, ri, E=E, k=k, act=O.RELU, moe_type=mt, dtype=O.F32, mode=O.MODE_EXACT)
    err = np.linalg.norm(got / scale - want / scale) / np.linalg.norm(want / scale)
    assert err <= REL, err


@pytest.mark.parametrize("tile", [0, 15, 16])
@pytest.mark.parametrize("mt", [O.QWEN3, O.NOMIC])
@pytest.mark.parametrize("T,H,I", [(70, 328, 136), (140, 76, 148), (33, 72, 264)])
def test_f32_non_finite_rows_among_finite_ones(tile, mt, T, H, I):
    """Rows of padding (all NaN, all infinite), a lone NaN or infinity anywhere
    along K, a NaN and an infinite weight: each sum is what f32 FMAs give, and
    rows without them stay as accurate as ever."""
    E, k = 2, 1
    x, G, U, D, rw, ri = moe_inputs(T, H, I, E, k, O.F32, 990 + T, mt)
    odd = {T - 1: np.nan, T - 2: np.nan, T - 3: np.inf, T - 4: -np.inf}
    for t, v in odd.items():
        x[t, :] = v
    lone = {0: (0, np.nan), 5: (H - 1, np.nan), 17: (H // 2, np.inf), 18: (H - 1, -np.inf), 19: (3, np.inf)}
    for t, (c, v) in lone.items():
        x[t, c] = v
    x[20, :] = 0.0
    G[0, H - 1, 7] = np.inf
    U[1, 2, 9] = np.nan
    G[1, H // 2, 3] = 0.0
    got = _forward(x, G, U, D, rw, ri, E, k, O.RELU, mt, tile).astype(np.float64)
    want = O.fused_moe(x, G, U, D, rw, ri, E=E, k=k, act=O.RELU, moe_type=mt, dtype=O.F32, mode=O.MODE_F32ACC)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf]) and np.array_equal(np.isinf(got), inf)
    fin = np.isfinite(want)
    assert np.linalg.norm(got[fin] - want[fin]) <= 1e-5 * np.linalg.norm(want[fin])


@pytest.mark.parametrize("T", [64, 2048])
def test_f32_padding_rows_of_nan_cost_little(T):
    """A sixteenth of the rows all NaN: at most three times the clean call (1.6
    and 1.1 times measured; recomputing whole blocks took 11 and 7.5 times)."""
    import torch

    H, I, E, k = 768, 3072, 8, 2
    gen = torch.Generator(device="cuda")
    gen.manual_seed(T)
    x, G, U = (torch.empty(s, device="cuda").normal_(0.0, d, generator=gen)
               for s, d in (((T, H), 1.0), ((E, H, I), 0.02), ((E, H, I), 0.02)))
    idx = torch.rand((T, E), device="cuda", generator=gen).argsort(1)[:, :k].to(torch.int32).contiguous()
    w = torch.full((T, k), 0.5, device="cuda")
    padded = x.clone()
    padded[-T // 16:] = float("nan")
    moe = candle_moe.FusedMoE.new(E, k, candle_moe.Activation.Gelu)

    def best(inp):
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            out = moe.forward(inp, G, U, None, w, idx, 1)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times), out

    clean, ref = best(x)
    slow, out = best(padded)
    assert torch.isnan(out[-T // 16:]).all()
    keep = slice(0, T - T // 16)
    assert (out[keep] - ref[keep]).norm() <= 1e-5 * ref[keep].norm()
    assert slow <= 3.0 * clean, (slow, clean)


@pytest.mark.parametrize("T,H,I,E,k,mt", [(1, 1024, 64, 1, 1, 0), (64, 1032, 72, 2, 1, 0), (17, 2056, 200, 3, 2, 1),
                                          (33, 4096, 8, 4, 2, 0), (256, 1096, 520, 8, 1, 0)])
def test_f32_decode_slices_of_few_blocks(T, H, I, E, k, mt):
    """K slices of the gate/up (fc1) GEMM over few 64-column blocks: K and column
    tails, empty slices. Bound as above, with one rounding per 16 k of both GEMMs
    and one per slice."""
    act = O.SILU if mt == 0 else O.GELU
    x, G, U, D, rw, ri = moe_inputs(T, H, I, E, k, O.F32, 920 + T, mt)
    got = _forward(x, G, U, D, rw, ri, E, k, act, mt, 0).astype(np.float64)
    want = O.fused_moe(x, G, U, D, rw, ri, E=E, k=k, act=act, moe_type=mt, dtype=O.F32, mode=O.MODE_EXACT)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= ((H + I) / 16 + 32) * 2.0 ** -24 + 4 * 2.0 ** -23, err
    assert np.array_equal(got, _forward(x, G, U, D, rw, ri, E, k, act, mt, 0))


@pytest.mark.parametrize("T,H,I,E", [(32, 4096, 1536, 1), (64, 1536, 768, 2), (64, 3432, 1160, 2)])
def test_f32_decode_of_few_experts_is_no_slower_than_tiles(T, H, I, E):
    """Few experts leave the decode kernels few items: sliced they take 0.6 to 0.85
    of the 32-row tiles' time; unsliced 1.4 to 1.6 times."""
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(T)
    x, G, U, D = (torch.empty(s, device="cuda").normal_(0.0, d, generator=gen)
                  for s, d in (((T, H), 1.0), ((E, H, I), 0.02), ((E, H, I), 0.02), ((E, I, H), 0.02)))
    idx = (torch.arange(T, device="cuda", dtype=torch.int32) % E).reshape(T, 1).contiguous()
    w = torch.ones((T, 1), device="cuda")
    moe = candle_moe.FusedMoE.new(E, 1, candle_moe.Activation.Silu)

    def best(tile):
        try:
            candle_moe.set_tile_policy(tile)
            times = []
            for _ in range(12):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                for _ in range(4):
                    moe.forward(x, G, U, D, w, idx, 0)
                b.record()
                torch.cuda.synchronize()
                times.append(a.elapsed_time(b))
            return min(times)
        finally:
            candle_moe.set_tile_policy(0)

    tiles, default = best(15), best(0)
    assert default <= 1.1 * tiles, (default, tiles)
