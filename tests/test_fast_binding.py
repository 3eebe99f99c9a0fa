"""candle_moe._fast against the ctypes route: the same descriptors, results and
errors for every form of tensor the entry points take or refuse."""
import ctypes
import os

import pytest
import torch

import candle_moe as cm

_REC = []
_TP = ctypes.POINTER(cm.CmTensor)


def _copy(p):
    d = cm.CmTensor()
    ctypes.memmove(ctypes.byref(d), p, ctypes.sizeof(d))
    return bytes(d)


@ctypes.CFUNCTYPE(ctypes.c_int, _TP, _TP, _TP, _TP, ctypes.c_void_p)
def _record(g, w, i, ei, stream):
    _REC.append(([_copy(t) for t in (g, w, i, ei)], stream))
    return 7


@pytest.fixture
def fast():
    cm.lib()
    if cm._native is None:
        pytest.skip("candle_moe._fast is not built")
    return cm._native


FORMS = {
    "2d": lambda: torch.zeros(5, 8),
    "transposed": lambda: torch.zeros(8, 5).t(),
    "strided": lambda: torch.zeros(5, 16)[:, ::2],
    "offset": lambda: torch.zeros(6, 8)[1:],
    "expanded": lambda: torch.zeros(1, 8).expand(5, 8),
    "scalar": lambda: torch.zeros(()),
    "empty": lambda: torch.zeros(0, 8),
    "rank4": lambda: torch.zeros(2, 3, 4, 5).permute(3, 1, 0, 2),
    "parameter": lambda: torch.nn.Parameter(torch.zeros(5, 8)),
    "f16": lambda: torch.zeros(5, 8, dtype=torch.float16),
    "bf16": lambda: torch.zeros(5, 8, dtype=torch.bfloat16),
    "i32": lambda: torch.zeros(5, 8, dtype=torch.int32),
    "u32": lambda: torch.zeros(5, 8, dtype=torch.uint32),
    "i64": lambda: torch.zeros(5, 8, dtype=torch.int64),
    "f64": lambda: torch.zeros(5, 8, dtype=torch.float64),
    "u8": lambda: torch.zeros(5, 8, dtype=torch.uint8),
    # left to the ctypes route
    "rank5": lambda: torch.zeros(1, 1, 1, 1, 1),
    "bool": lambda: torch.zeros(5, 8, dtype=torch.bool),
    "sparse": lambda: torch.zeros(5, 8).to_sparse(),
    "meta": lambda: torch.zeros(5, 8, device="meta"),
    "none": lambda: None,
}
LEFT = {"rank5", "bool", "sparse", "meta", "none"}


@pytest.mark.parametrize("name", list(FORMS))
def test_descriptors(fast, name):
    """The descriptors the C entry receives are describe()'s, byte for byte."""
    t = FORMS[name]()
    L = cm.lib()
    addr = lambda fn: ctypes.cast(fn, ctypes.c_void_p).value  # noqa: E731
    rest = [addr(L.candle_moe_fused_moe_forward), addr(L.candle_moe_router_topk), addr(L.candle_moe_fused_moe_fp8),
            addr(L.candle_moe_fused_moe_packed), torch._C._cuda_getCurrentRawStream]
    _REC.clear()
    fast.bind(addr(_record), *rest)
    try:
        got = fast.topk(t, torch.zeros(5, 2), t, torch.zeros(5, 2, dtype=torch.int32))
    finally:
        fast.bind(addr(L.candle_moe_apply_topk_softmax_inplace), *rest)
    if name in LEFT:
        assert got is None and not _REC
        return
    assert got == 7 and len(_REC) == 1
    descs, stream = _REC[0]
    want = bytes(cm.describe(t))
    assert descs[0] == want and descs[2] == want and not stream


def test_wrong_arguments(fast):
    x = torch.zeros(2, 2)
    with pytest.raises(TypeError):
        fast.topk(x, x, x)
    # values the ctypes route converts or rejects
    assert fast.forward(4, 2, 0, x, x, x, None, x, x, 2) is None
    assert fast.forward(4, 2, 0, x, x, x, None, x, x, 0.0) is None
    assert fast.forward(1 << 80, 2, 0, x, x, x, None, x, x, 0) is None


def _both(monkeypatch, f):
    """f() through the binding and through ctypes: results, or the error raised."""
    out = []
    for fast in (cm._native, None):
        monkeypatch.setattr(cm, "_native", fast)
        try:
            out.append(f())
        except Exception as e:  # noqa: BLE001
            out.append((type(e), str(e)))
    return out


def _same(a, b):
    if isinstance(a, torch.Tensor):
        return isinstance(b, torch.Tensor) and a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)
    return a == b


def _moe(dt=torch.bfloat16, T=5, H=64, I=32, E=4, k=2):
    g = torch.Generator().manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g).to(dt).cuda()  # noqa: E731
    return dict(x=r(T, H), gate=r(E, H, I), up=r(E, H, I), down=r(E, I, H), rw=r(T, k).float(),
                ix=torch.randint(0, E, (T, k), generator=g, dtype=torch.int32).cuda())


BREAK = {
    "as is": lambda a: None,
    "f32": lambda a: a.update({n: a[n].float() for n in ("x", "gate", "up", "down")}),
    "strided x": lambda a: a.update(x=a["x"].repeat(1, 2)[:, ::2]),
    "transposed down": lambda a: a.update(down=a["down"].transpose(1, 2).contiguous().transpose(1, 2)),
    "cpu weights": lambda a: a.update(gate=a["gate"].cpu()),
    "cpu input": lambda a: a.update(x=a["x"].cpu()),
    "1-d input": lambda a: a.update(x=a["x"][0]),
    "f16 routing": lambda a: a.update(rw=a["rw"].half()),
    "i64 indices": lambda a: a.update(ix=a["ix"].long()),
    "u32 indices": lambda a: a.update(ix=a["ix"].view(torch.uint32)),
    "few indices": lambda a: a.update(ix=a["ix"][:-1]),
    "no tokens": lambda a: a.update(x=a["x"][:0], rw=a["rw"][:0], ix=a["ix"][:0]),
    "no down": lambda a: a.update(down=None),
    "mixed": lambda a: a.update(up=a["up"].half()),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(BREAK))
def test_routes_agree(fast, monkeypatch, name):
    a = _moe()
    BREAK[name](a)
    m = cm.FusedMoE(4, 2, cm.Activation.Silu)

    def forward():
        return m.forward(a["x"], a["gate"], a["up"], a["down"], a["rw"], a["ix"], 0)

    def prepared(fp8):
        out = torch.zeros_like(a["x"])
        t = lambda w: w if w is None else w.transpose(1, 2).contiguous()  # noqa: E731
        w = [t(a[n]) for n in ("gate", "up", "down")]
        if fp8:
            q = [cm.quantize_fp8(v.cuda(), False) if v is not None else (None, None) for v in w]
            cm.fused_moe_fp8(a["x"], *[c for c, _ in q], *[s for _, s in q], a["rw"], a["ix"], out, 4, 2)
        else:
            cm.fused_moe_packed(a["x"], *w, a["rw"], a["ix"], out, 4, 2)
        return out

    def router():
        x = a["x"].cuda()  # (the ctypes route takes the tensors' devices as given)
        T = x.shape[0]
        o = [torch.zeros(T, 2, device="cuda"), a["ix"].clone(), torch.zeros_like(a["ix"])]
        cm.router_topk(x, x.new_ones(4, x.shape[-1]), *o)
        return torch.cat([t.float() for t in o])

    for f in (forward, lambda: prepared(False), lambda: prepared(True), router):
        got, want = _both(monkeypatch, f)
        assert _same(got, want), (name, got, want)


@pytest.mark.gpu
def test_stream(fast):
    """Calls go to the current stream of the input's device."""
    a = _moe()
    s = torch.cuda.Stream()
    m = cm.FusedMoE(4, 2, cm.Activation.Silu)
    call = lambda: m.forward(a["x"], a["gate"], a["up"], a["down"], a["rw"], a["ix"], 0)  # noqa: E731
    want = call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        call()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        out = call()
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def _calls():
    """Every entry point with its tensors, small and valid."""
    T, H, I, E, k = 3, 64, 64, 4, 2
    bf = dict(dtype=torch.bfloat16, device="cuda")
    f32, i32 = dict(device="cuda"), dict(dtype=torch.int32, device="cuda")
    w, idx, te = torch.full((T, k), 0.5, **f32), torch.zeros(T, k, **i32), torch.zeros(T, k, **i32)
    x, out, G = torch.ones(T, H, **bf), torch.zeros(T, H, **bf), torch.ones(E, H, I, **bf)
    u8 = dict(dtype=torch.uint8, device="cuda")
    q, sc = torch.zeros(E, I, H, **u8), torch.ones(E, I, **f32)
    moe = cm.FusedMoE.new(E, k, cm.Activation.Silu)
    return {
        "topk": (cm.apply_topk_softmax_inplace, [torch.zeros(T, E, **f32), w, idx, te], ()),
        "router": (cm.router_topk, [x, torch.ones(E, H, **bf), w, idx, te], ()),
        "forward": (lambda *a: moe.forward(*a, 0), [x, G, G.clone(), G.clone(), w, idx], ()),
        "packed": (cm.fused_moe_packed, [x, G, G.clone(), G.clone(), w, idx, out], (E, k, 0, 0)),
        "fp8": (cm.fused_moe_fp8, [x, q, q.clone(), q.clone(), sc, sc.clone(), sc.clone(), w, idx, out], (E, k, 0, 0)),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["topk", "router", "forward", "packed", "fp8"])
def test_tensor_that_refuses_its_pointer(name):
    """A tensor whose data pointer must not be read raises, as on the ctypes
    route, whichever argument it is; the interpreter lock is held by then."""
    for i in range(len(_calls()[name][1])):
        fn, tensors, rest = _calls()[name]
        tensors[i] = tensors[i].clone()
        torch._C._set_throw_on_mutable_data_ptr(tensors[i])
        with pytest.raises(RuntimeError, match="data pointer"):
            fn(*tensors, *rest)
    fn, tensors, rest = _calls()[name]
    fn(*tensors, *rest)
    torch.cuda.synchronize()


def test_the_library_loads_without_torch():
    """lib() alone does not import torch; the binding follows once it is there."""
    import subprocess
    import sys

    code = ("import sys, candle_moe as cm; cm.lib(); cm.lib(); assert 'torch' not in sys.modules; "
            "assert cm._native is None; import torch; cm.lib(); "
            "import importlib.util as u; "
            "assert (cm._native is not None) == (u.find_spec('candle_moe._fast') is not None)")
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300,
                   env=dict(os.environ, PYTHONPATH=os.path.dirname(os.path.dirname(cm.__file__))))
