"""Captured graphs hold the address of their stream's workspace: a larger eager
call on that stream, which replaces it, leaves the memory to them."""
import ctypes

import numpy as np
import pytest
import torch

import candle_moe
import oracle as O
from helpers import assert_close, from_dev, moe_inputs, to_dev
from test_gpu_router import quantized

pytestmark = pytest.mark.gpu


def pool_bytes():
    """Bytes in use in the device's stream-ordered memory pool (the workspaces')."""
    candle_moe.lib()
    path = next(p for p in (ln.split()[-1] for ln in open("/proc/self/maps")) if "libamdhip64" in p)
    hip = ctypes.CDLL(path)
    pool, used = ctypes.c_void_p(), ctypes.c_uint64()
    assert hip.hipDeviceGetDefaultMemPool(ctypes.byref(pool), 0) == 0
    assert hip.hipMemPoolGetAttribute(pool, 7, ctypes.byref(used)) == 0  # hipMemPoolAttrUsedMemCurrent
    return used.value


def outputs(T, k):
    return [torch.zeros((T, k), dtype=d, device="cuda") for d in (torch.float32, torch.int32, torch.int32)]


def router_case(T, H, E, k, dt):
    x, w = (O.to_dtype(quantized(s, d, T + n), dt) for s, d, n in (((T, H), 8.0, 1), ((E, H), 64.0, 2)))
    want = O.topk_softmax(O.router_logits(x, w, dt), k)
    return to_dev(x, dt), to_dev(w, dt), want


def captured(s, call):
    """call() once eagerly, then captured, on stream s."""
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call()
    return g


def test_router_graph_outlives_a_larger_call():
    H, E, k, dt = 2048, 128, 8, O.BF16
    candle_moe.trim_workspaces()
    empty = pool_bytes()
    s = torch.cuda.Stream()
    x1, w1, (ww, wi, _) = router_case(1, H, E, k, dt)
    out = outputs(1, k)
    g = captured(s, lambda: candle_moe.router_topk(x1, w1, *out))
    small = pool_bytes()
    assert small > empty
    # 1000 tokens need 4 MB of partials: another buffer, beside the graph's
    x2, w2, (_, wi2, _) = router_case(1000, H, E, k, dt)
    out2 = outputs(1000, k)
    s.wait_stream(torch.cuda.current_stream())
    for _ in range(3):
        with torch.cuda.stream(s):
            candle_moe.router_topk(x2, w2, *out2)
        torch.cuda.synchronize()
        assert pool_bytes() >= small + 1000 * E * 4 * 2, "the graph's buffer was released"
        for t in out:
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(from_dev(out[1]).astype(np.uint32), wi)
        np.testing.assert_allclose(from_dev(out[0]), ww, rtol=1e-6, atol=0)
        assert np.array_equal(from_dev(out2[1]).astype(np.uint32), wi2)
    del g
    candle_moe.trim_workspaces()
    assert pool_bytes() == empty


def test_layer_graph_outlives_a_larger_call():
    H, I, E, k, dt = 256, 128, 4, 2, O.BF16
    candle_moe.trim_workspaces()
    empty = pool_bytes()
    s = torch.cuda.Stream()

    def case(T):
        x, G, U, D, rw, ri = moe_inputs(T, H, I, E, k, dt, 40 + T, O.QWEN3)
        want = O.fused_moe(x, G, U, D, rw, ri, E=E, k=k, act=O.SILU, moe_type=0, dtype=dt, mode=O.MODE_F32ACC)
        return [to_dev(a, dt) for a in (x, G, U, D)] + [to_dev(rw), to_dev(ri)], np.asarray(want, dtype=np.float64)

    moe = candle_moe.FusedMoE.new(E, k, candle_moe.Activation.Silu)
    small, want = case(3)
    keep = {}

    def call():
        keep["out"] = moe.forward(*small, 0)

    g = captured(s, call)
    before = pool_bytes()
    assert before > empty
    large, want2 = case(4000)
    s.wait_stream(torch.cuda.current_stream())
    for _ in range(2):
        with torch.cuda.stream(s):
            out2 = moe.forward(*large, 0)
        torch.cuda.synchronize()
        assert pool_bytes() >= before + 4000 * k * I * 2, "the graph's buffer was released"
        keep["out"].zero_()
        g.replay()
        torch.cuda.synchronize()
        assert_close(from_dev(keep["out"]), want, 2e-2)
        assert_close(from_dev(out2), want2, 2e-2)
    del g
    candle_moe.trim_workspaces()
    assert pool_bytes() == empty


def forward_case(T, H, I, E, k, dt):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(T)
    x, G, U, D = (torch.empty(s, dtype=dt, device="cuda").normal_(0.0, d, generator=gen)
                  for s, d in (((T, H), 1.0), ((E, H, I), 0.02), ((E, H, I), 0.02), ((E, I, H), 0.02)))
    idx = torch.rand((T, E), device="cuda", generator=gen).argsort(1)[:, :k].to(torch.int32).contiguous()
    return x, G, U, D, torch.full((T, k), 1.0 / k, device="cuda"), idx


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,I,E,k,most,fewer", [(2048, 768, 128, 8, 6, (1, 5)), (4096, 512, 8, 2, 2, (1,)),
                                                (1280, 1888, 64, 2, 120, (3, 17, 64, 99)),
                                                (768, 3072, 8, 2, 300, (128, 129, 200))])
@pytest.mark.parametrize("pregrown", [False, True])
def test_one_call_of_the_largest_size(H, I, E, k, most, fewer, dt, pregrown):
    """After one eager call the smaller batches of the layer can be captured,
    also where another call's workspace was there and held that eager call."""
    candle_moe.trim_workspaces()
    s = torch.cuda.Stream()
    moe = candle_moe.FusedMoE.new(E, k, candle_moe.Activation.Silu)
    x, G, U, D, w, idx = forward_case(most, H, I, E, k, dt)
    xr, wr, _ = router_case(1000, 2048, 128, 8, O.BF16)
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        if pregrown:
            candle_moe.router_topk(xr, wr, *outputs(1000, 8))
        moe.forward(x, G, U, D, w, idx, 0)
    torch.cuda.synchronize()
    for T in fewer:
        args = x[:T].contiguous(), G, U, D, w[:T].contiguous(), idx[:T].contiguous(), 0
        want = moe.forward(*args)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = moe.forward(*args)
        for _ in range(2):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            # (K splits of few tiles meet in f32 atomics: the last bits may differ)
            assert (out - want).norm() <= (1e-2 if dt is torch.bfloat16 else 1e-5) * want.norm(), T
        del g


@pytest.mark.parametrize("most,fewer", [(129, 128), (4099, 200), (1000, 256)])
def test_router_after_a_larger_call(most, fewer):
    H, E, k, dt = 2048, 128, 8, O.BF16
    candle_moe.trim_workspaces()
    s = torch.cuda.Stream()
    xl, wl, _ = router_case(most, H, E, k, dt)
    x, w, (ww, wi, _) = router_case(fewer, H, E, k, dt)
    small = forward_case(1, 256, 128, 4, 2, torch.bfloat16)
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):  # (the layer's workspace of 1 MiB is there first)
        candle_moe.FusedMoE.new(4, 2, candle_moe.Activation.Silu).forward(*small, 0)
        candle_moe.router_topk(xl, wl, *outputs(most, k))
    torch.cuda.synchronize()
    out = outputs(fewer, k)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        candle_moe.router_topk(x, w, *out)
    for _ in range(2):
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(from_dev(out[1]).astype(np.uint32), wi)
        np.testing.assert_allclose(from_dev(out[0]), ww, rtol=1e-6, atol=0)
