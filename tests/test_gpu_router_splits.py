"""router_topk past 256 tokens: K splits over workgroups where they pay, the same
sums inside one workgroup per tile under graph capture, one pass otherwise; stages
of two K tiles with odd tile counts and K tails. Inputs whose sums are exact in f32 (small
integers over powers of two), so every form gives the oracle's indices bit for
bit and its weights within 1e-6 (f32 exp and quotient, as in
tests/test_gpu_router.py)."""
import numpy as np
import pytest
import torch

import candle_moe
import oracle as O
from helpers import from_dev, to_dev
from test_gpu_router import quantized, run_fused

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [O.BF16, O.F16])
@pytest.mark.parametrize("T,H,E,k", [
    (257, 2048, 128, 8), (1023, 1608, 65, 8), (2080, 2048, 100, 4),   # split: ragged tiles, K tail, few splits
    (300, 4096, 64, 6), (4095, 4096, 33, 2),
    (4097, 2048, 128, 8), (300, 1536, 128, 8),                        # one pass: too many tiles, too little K
    (300, 8, 128, 8), (300, 72, 64, 2), (300, 136, 40, 2), (300, 320, 128, 2),  # K tiles 1, 2, 3, 5
    (8193, 72, 128, 8), (8193, 72, 64, 8),                            # 64 tokens per workgroup from here (E > 64)
])
def test_exact(dt, T, H, E, k):
    x = O.to_dtype(quantized((T, H), 8.0, T + H), dt)
    w = O.to_dtype(quantized((E, H), 64.0, E + k), dt)
    gw, gi, ge = run_fused(x, w, k, dt)
    ww, wi, we = O.topk_softmax(O.router_logits(x, w, dt), k)
    assert np.array_equal(gi, wi) and np.array_equal(ge, we)
    np.testing.assert_allclose(gw, ww, rtol=1e-6, atol=0)


@pytest.mark.parametrize("warm", [False, True])
def test_capture(warm):
    """Captured on a stream without a workspace, and on one that has it."""
    T, H, E, k, dt = 1000, 2048, 128, 8, O.BF16
    x, w = (O.to_dtype(quantized(s, d, n), dt) for s, d, n in (((T, H), 8.0, 1), ((E, H), 64.0, 2)))
    ww, wi, _ = O.topk_softmax(O.router_logits(x, w, dt), k)
    xt, wt = to_dev(x, dt), to_dev(w, dt)
    out = [torch.zeros((T, k), dtype=d, device="cuda") for d in (torch.float32, torch.int32, torch.int32)]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    if warm:
        with torch.cuda.stream(s):
            candle_moe.router_topk(xt, wt, *out)
    else:
        candle_moe.trim_workspaces()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        candle_moe.router_topk(xt, wt, *out)
    for _ in range(3):
        for t in out:
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(from_dev(out[1]).astype(np.uint32), wi)
        np.testing.assert_allclose(from_dev(out[0]), ww, rtol=1e-6, atol=0)
        run_fused(x, w, k, dt)  # the program's own work between replays


@pytest.mark.parametrize("T,H,E,k,dt", [
    (257, 2048, 128, 8, torch.bfloat16), (1000, 2056, 128, 8, torch.bfloat16),  # the exact and the f32 softmax
    (2000, 2048, 128, 20, torch.float16), (700, 2880, 100, 4, torch.bfloat16),
    (3283, 4096, 64, 8, torch.bfloat16), (1001, 4096, 40, 2, torch.float16),
    (290, 1736, 65, 3, torch.float16),
])
def test_capture_gives_the_eager_bits(T, H, E, k, dt):
    """Logits of every rounding: the captured call adds the K ranges up in the
    order in which the eager one does and takes the same softmax."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(T + H)
    x = torch.empty((T, H), dtype=dt, device="cuda").normal_(0.0, 1.0, generator=gen)
    w = torch.empty((E, H), dtype=dt, device="cuda").normal_(0.0, 0.02, generator=gen)
    eager, out = ([torch.zeros((T, k), dtype=d, device="cuda") for d in (torch.float32, torch.int32, torch.int32)]
                  for _ in range(2))
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        candle_moe.router_topk(x, w, *out)
    for _ in range(3):
        for t in out:
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        candle_moe.router_topk(x, w, *eager)  # the program's own work between replays
        for a, b in zip(eager, out):
            assert torch.equal(a, b)
