"""Performance cases: the calls a program that serves MoE models makes.

Each case is one call or one short sequence of calls through the package's
public entry points, on inputs that are resident on the GPU:

  topk     apply_topk_softmax_inplace over a batch of router logits
  router   router_topk: the router GEMM fused with softmax and top-k
  layer    a whole MoE layer: apply_topk_softmax_inplace, then FusedMoE.forward
  fp8      the same layer over fp8 expert weights (fused_moe_fp8 adds into its
           output, so the caller clears it first)
  packed   the same layer over pre-packed 16-bit weights (fused_moe_packed)

The model sizes are the repository's own: Qwen3 (H 4096, I 1536, 8 experts,
top 2), Qwen3-30B-A3B (H 2048, I 768, 128 experts, top 8) and Nomic (H 768,
I 3072, 8 experts, top 2, GELU); drawn cases add ragged generic ones.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "candle-moe_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import candle_moe  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}
QWEN3 = dict(H=4096, I=1536, E=8, k=2, act="silu", moe_type=0)
Q30B = dict(H=2048, I=768, E=128, k=8, act="silu", moe_type=0)
NOMIC = dict(H=768, I=3072, E=8, k=2, act="gelu", moe_type=1)


def _moe(kind, name, model, T, dtype, skew=False):
    c = dict(kind=kind, T=T, dtype=dtype, skew=skew, **model)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one token of a chat decode step: the router alone, latency only
        dict(name="router_decode_1", kind="router", T=1, H=2048, E=128, k=8, dtype="bf16"),
        # the router of a ragged prefill chunk
        dict(name="router_prefill_4099", kind="router", T=4099, H=2048, E=128, k=8, dtype="bf16"),
        # logits computed by the caller, a full prefill batch
        dict(name="topk_32768x128", kind="topk", T=32768, E=128, k=8, dtype="f32"),
        # single-user decode: a few experts' weights, cold
        _moe("layer", "q30b_decode_1", Q30B, 1, "bf16"),
        # a small decode batch: every expert's weights once
        _moe("layer", "qwen3_decode_8", QWEN3, 8, "bf16"),
        # the same served from fp8 weights
        _moe("fp8", "qwen3_fp8_decode_16", QWEN3, 16, "bf16"),
        # a ragged chunk of a mixed prefill / decode batch
        _moe("layer", "qwen3_chunk_500", QWEN3, 500, "bf16"),
        # a prefill chunk over many small experts
        _moe("layer", "q30b_prefill_4096", Q30B, 4096, "bf16"),
        # the largest prefill batch
        _moe("layer", "qwen3_prefill_32768", QWEN3, 32768, "bf16"),
        # an embedding model in f32: a few queries, then a batch of documents
        _moe("layer", "nomic_f32_64", NOMIC, 64, "f32"),
        _moe("layer", "nomic_f32_4096", NOMIC, 4096, "f32"),
        # the embedding model in f16, a ragged batch of documents
        _moe("layer", "nomic_f16_8191", NOMIC, 8191, "f16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(2 ** rng.uniform(math.log2(lo), math.log2(hi))))))


def draw(rng):
    kind = rng.choice(["topk", "router", "layer", "layer", "layer", "layer", "layer", "layer", "fp8", "packed"])
    if kind == "topk":
        E = rng.choice([8, 16, 32, 60, 64, 100, 128, 256])
        return dict(kind=kind, T=_log_int(rng, 1, 32768), E=E, k=rng.randint(1, min(8, E)),
                    dtype=rng.choice(["f32", "f32", "f16", "bf16"]))
    if kind == "router":
        E = rng.choice([8, 16, 32, 60, 64, 128])
        return dict(kind=kind, T=_log_int(rng, 1, 32768), H=rng.choice([768, 2048, 2880, 4096]), E=E,
                    k=rng.randint(1, min(8, E)), dtype=rng.choice(["bf16", "bf16", "f16"]))
    model = rng.choice([QWEN3, Q30B, NOMIC, None])
    if model is None:
        step = 16 if kind == "fp8" else 8
        E = rng.choice([4, 8, 16, 32, 60, 64])
        model = dict(H=step * rng.randint(256 // step, 4096 // step), I=step * rng.randint(256 // step, 2048 // step),
                     E=E, k=rng.randint(1, min(8, E)), act=rng.choice(["silu", "gelu", "relu"]),
                     moe_type=rng.randint(0, 1))
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"] if kind == "layer" else ["bf16", "f16"])
    T = _log_int(rng, 1, 32768)
    # no more work than the largest listed case of the same type
    per_token = model["k"] * 2 * (3 if model["moe_type"] == 0 else 2) * model["H"] * model["I"]
    most = 7.7e10 if dtype == "f32" else 1.5e12
    T = max(1, min(T, int(most / per_token)))
    return _moe(kind, None, model, T, dtype, skew=rng.random() < 0.25)


def _normal(shape, dtype, gen, std=1.0):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)


def _inputs(case, seed):
    """The tensors of a case from its seed alone (no call into the package)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 7919 + 17)
    dt = DTYPES[case["dtype"]]
    T, E = case["T"], case["E"]
    if case["kind"] == "topk":
        return {"logits": _normal((T, E), dt, gen)}
    H = case["H"]
    if case["kind"] == "router":
        return {"x": _normal((T, H), dt, gen), "w": _normal((E, H), dt, gen, 0.02)}
    I = case["I"]
    logits = _normal((T, E), torch.float32, gen)
    if case["skew"]:  # some experts are favoured, as trained routers do
        logits += 1.0 / (1.0 + torch.arange(E, device="cuda", dtype=torch.float32))[torch.randperm(E, generator=gen, device="cuda")]
    s = {"logits": logits, "x": _normal((T, H), dt, gen), "gate": _normal((E, H, I), dt, gen, 0.02)}
    if case["moe_type"] == 0:
        s["up"] = _normal((E, H, I), dt, gen, 0.02)
        s["down"] = _normal((E, I, H), dt, gen, 0.02)
    else:  # fc2 is [E, H, I] in the up position
        s["up"] = _normal((E, H, I), dt, gen, 0.02)
        s["down"] = None
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    T, k = case["T"], case["k"]
    wt = DTYPES[case["dtype"]] if case["kind"] == "topk" else torch.float32
    s["weights"] = torch.empty((T, k), dtype=wt, device="cuda")
    s["indices"] = torch.empty((T, k), dtype=torch.int32, device="cuda")
    s["token_expert"] = torch.empty((T, k), dtype=torch.int32, device="cuda")
    s["case"] = case
    if case["kind"] in ("layer", "fp8", "packed"):
        act = {"silu": candle_moe.Activation.Silu, "gelu": candle_moe.Activation.Gelu,
               "relu": candle_moe.Activation.Relu}[case["act"]]
        s["act"] = act
        s["moe"] = candle_moe.FusedMoE.new(case["E"], k, act)
        s["out"] = torch.empty_like(s["x"])
    if case["kind"] == "packed":
        s["gate"] = candle_moe.pack_weights(s["gate"])
        if case["moe_type"] == 0:
            s["up"] = candle_moe.pack_weights(s["up"])
            s["down"] = candle_moe.pack_weights(s["down"])
    if case["kind"] == "fp8":
        kn = case["moe_type"] == 0
        s["gate"], s["gate_s"] = candle_moe.quantize_fp8(s["gate"], True)
        s["up"], s["up_s"] = candle_moe.quantize_fp8(s["up"], kn)
        s["down_s"] = None
        if kn:
            s["down"], s["down_s"] = candle_moe.quantize_fp8(s["down"], True)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "router":
        candle_moe.router_topk(s["x"], s["w"], s["weights"], s["indices"], s["token_expert"])
        return [s["weights"], s["indices"], s["token_expert"]]
    candle_moe.apply_topk_softmax_inplace(s["logits"], s["weights"], s["indices"], s["token_expert"])
    if kind == "topk":
        return [s["weights"], s["indices"], s["token_expert"]]
    if kind == "layer":
        out = s["moe"].forward(s["x"], s["gate"], s["up"], s["down"], s["weights"], s["indices"], c["moe_type"])
    elif kind == "fp8":
        out = s["out"].zero_()
        candle_moe.fused_moe_fp8(s["x"], s["gate"], s["up"], s["down"], s["gate_s"], s["up_s"], s["down_s"],
                                 s["weights"], s["indices"], out, c["E"], c["k"], int(s["act"]), c["moe_type"])
    else:
        out = s["out"].zero_()
        candle_moe.fused_moe_packed(s["x"], s["gate"], s["up"], s["down"], s["weights"], s["indices"], out,
                                    c["E"], c["k"], int(s["act"]), c["moe_type"])
    return [out, s["weights"], s["indices"], s["token_expert"]]


def work(case):
    T, E, k, s = case["T"], case["E"], case["k"], SIZE[case["dtype"]]
    if case["kind"] == "topk":
        return {"bytes": T * E * s + T * k * (s + 8), "flops": 0}
    if case["kind"] == "router":
        H = case["H"]
        return {"bytes": (T + E) * H * s + T * k * 12, "flops": 2 * T * E * H}
    H, I = case["H"], case["I"]
    m = 3 if case["moe_type"] == 0 else 2
    touched = E * (1.0 - (1.0 - k / E) ** T)  # experts with a token, routing at random
    ws = 1 if case["kind"] == "fp8" else s
    scales = touched * (2 * I + H) * 4 if case["kind"] == "fp8" else 0
    return {"bytes": touched * m * H * I * ws + scales + 2 * T * H * s + T * E * 4 + T * k * 12,
            "flops": 2.0 * m * T * k * H * I}


def tolerance(case):
    # Four times what separates the path from the same sums in another order
    # or in 64 bits. Indices are whole values: logits in f32 (or given) leave
    # no ties to speak of; a router GEMM's logits are rounded to 16 bits, so
    # sums in another order can move one to its neighbour.
    if case["kind"] == "topk":
        return {"rel": 2e-6 if case["dtype"] == "f32" else 8e-3, "differ": 1e-4}
    if case["kind"] == "router":
        return {"rel": 4e-3 if case["dtype"] == "bf16" else 1e-3, "differ": 2e-3}
    return {"rel": {"bf16": 1e-2, "f16": 2e-3, "f32": 6e-6}[case["dtype"]], "differ": 1e-4}


def _exact_topk(logits, k):
    T = logits.shape[0]
    p = torch.softmax(logits.double(), dim=-1)
    w, i = torch.sort(p.float(), dim=-1, descending=True, stable=True)
    i = i[:, :k]
    w = torch.gather(p, 1, i)
    te = torch.arange(k, device="cuda").unsqueeze(0) * T + torch.arange(T, device="cuda").unsqueeze(1)
    return w, i.to(torch.int32), te.to(torch.int32)


def _fp8(w):
    """[E, N, K] weights as their fp8 e4m3 codes stand for them, in 64 bits."""
    w = w.float()
    s = w.abs().amax(dim=-1, keepdim=True)
    s = s / torch.full_like(s, 448.0)  # (by a number, torch multiplies by its reciprocal)
    s = torch.where(s > 0, s, torch.ones_like(s))
    return (w / s).to(torch.float8_e4m3fn).double() * s.double()


def exact(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "topk":
        return list(_exact_topk(s["logits"], case["k"]))
    if case["kind"] == "router":
        logits = (s["x"].double() @ s["w"].double().t()).to(DTYPES[case["dtype"]])
        return list(_exact_topk(logits, case["k"]))
    w, idx, te = _exact_topk(s["logits"], case["k"])
    x = s["x"].double()
    out = torch.zeros_like(x)
    f8 = case["kind"] == "fp8"

    def nk(t, e, kn):  # one expert's weight as [N, K]
        t = t[e].t() if kn else t[e]
        return _fp8(t) if f8 else t.double()

    act = {"silu": torch.nn.functional.silu, "relu": torch.relu,
           "gelu": lambda v: torch.nn.functional.gelu(v, approximate="tanh")}[case["act"]]
    qwen = case["moe_type"] == 0
    for e in range(case["E"]):
        t, j = torch.nonzero(idx == e, as_tuple=True)
        if t.numel() == 0:
            continue
        xe = x[t]
        h = act(xe @ nk(s["gate"], e, True).t().contiguous())
        if qwen:
            h = h * (xe @ nk(s["up"], e, True).t().contiguous())
            y = h @ nk(s["down"], e, True).t().contiguous()
        else:
            y = h @ nk(s["up"], e, False).t().contiguous()
        out.index_add_(0, t, y * w[t, j].unsqueeze(1))
    return [out, w, idx, te]
