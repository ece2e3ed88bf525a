"""The measured work: what a program built on this library has it do.

Every case goes through the public entry points (MoeLayer, MoeStack, or the C
ABI's operator entries where no class wraps them).  Four kinds of call:

  forward  one MoE layer on T tokens (router, dispatch, experts, combine)
  block    one decoder-block MLP half: RMSNorm, the layer, the residual add
  stack    several blocks in one call, as a decode step runs them
  gemv     the W4A8 operator pair: quantize the activations, INT4 x int8 GEMV

over batch-1 decode, batched decode, speculative verify, ragged and full
prefill chunks and calls of several chunks, uniform and Zipf routing, both
precisions, both scale types, both norm forms, with and without shared expert
and gate.
"""
import ctypes as C
import math

import numpy as np
import torch

from ainfer_amd import _lib as L
from ainfer_amd.moe import MoeLayer, MoeStack, make_input
from ainfer_amd.synthetic import MoeConfig

DEV = "cuda"
EPS = 1e-6


def _layer_case(name, kind, dims, tokens, precision="w4a16", scales="fp16", norm="plain",
                zipf=0.0, layers=1, gate=True):
    hidden, experts, top_k, inter, shared = dims
    return dict(name=name, kind=kind, hidden=hidden, experts=experts, top_k=top_k, inter=inter,
                shared=shared, tokens=tokens, precision=precision, scales=scales, norm=norm,
                zipf=zipf, layers=layers, gate=gate)


# the benchmark's layer dimensions: H, E, k, I, I of the shared expert
SMALL = (1024, 64, 8, 256, 256)
MID = (2048, 512, 10, 512, 512)
LARGE = (4096, 512, 10, 1024, 1024)
# no power of two anywhere: 20 and 7 quantization groups, a wide shared expert
ODD = (2560, 96, 6, 896, 1792)


def listed():
    return [
        # the smallest call: one token through a small block (all latency)
        _layer_case("block_small_T1", "block", SMALL, 1),
        # batch-1 decode, the benchmark's headline step (4 of its 60 blocks)
        _layer_case("stack_large_T1", "stack", LARGE, 1, layers=4),
        # the same step for a batch of 8 sequences
        _layer_case("stack_large_T8", "stack", LARGE, 8, layers=4),
        # batch-16 decode of a mid-size layer
        _layer_case("forward_mid_T16", "forward", MID, 16),
        # speculative-decode verify: 64 tokens in one call
        _layer_case("forward_large_T64", "forward", LARGE, 64),
        # a ragged prompt on odd dimensions, bf16 scales, (1 + w) norm, no gate
        _layer_case("block_odd_T301", "block", ODD, 301, scales="bf16", norm="one_plus",
                    gate=False),
        # a partly filled prefill chunk, balanced routing
        _layer_case("block_mid_T1500", "block", MID, 1500),
        # a full prefill chunk, popular and rare experts
        _layer_case("forward_mid_T4096_zipf", "forward", MID, 4096, zipf=1.1),
        # a long prompt in one call (several chunks), balanced routing
        _layer_case("forward_mid_T16384", "forward", MID, 16384),
        # batch-1 decode in the W4A8 precision
        _layer_case("w4a8_stack_large_T1", "stack", LARGE, 1, precision="w4a8", layers=4),
        # a prompt in the W4A8 precision
        _layer_case("w4a8_forward_mid_T512", "forward", MID, 512, precision="w4a8"),
        # the W4A8 operators alone, the benchmark's GEMV shape
        dict(name="w4a8_gemv_T1", kind="gemv", rows=17408, cols=5120, tokens=1, scales="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _even_or_small(groups):
    # the layer takes hidden sizes of up to 15 groups, or an even number up to 32
    return groups if groups <= 15 or groups % 2 == 0 else groups - 1


def draw(rng):
    if rng.random() < 0.08:
        return dict(kind="gemv", rows=_log_int(rng, 200, 20000), cols=128 * _log_int(rng, 2, 64),
                    tokens=rng.choice((1, 1, 1, 2, 5, 16)), scales=rng.choice(("bf16", "fp16")))
    precision = rng.choice(("w4a16", "w4a16", "w4a16", "w4a8"))
    biggest = max(work(c)["flops"] for c in listed())
    while True:
        if rng.random() < 0.5:
            dims = rng.choice((SMALL, MID, LARGE, ODD))
        else:
            experts = _log_int(rng, 8, 512)
            inter = 128 * rng.randint(1, 10)
            dims = (128 * _even_or_small(rng.randint(6, 32)), experts,
                    rng.randint(1, min(experts, 12)), inter, rng.choice((0, inter, inter, 2 * inter)))
            if dims[4] > 4096:
                continue
        top = 1024 if precision == "w4a8" else 16384
        # half of all calls are decode steps
        tokens = _log_int(rng, 1, 24) if rng.random() < 0.5 else _log_int(rng, 16, top)
        kind = rng.choice(("forward", "block")) if tokens > 16 else rng.choice(
            ("forward", "block", "stack"))
        case = _layer_case("", kind, dims, tokens, precision=precision,
                           scales=rng.choice(("fp16", "fp16", "bf16")),
                           norm=rng.choice(("plain", "one_plus")),
                           zipf=rng.choice((0.0, 0.0, 1.1)),
                           layers=rng.randint(2, 4) if kind == "stack" else 1,
                           gate=rng.random() < 0.8)
        del case["name"]
        # no more than the largest listed case, in arithmetic and in weights
        w = work(case)
        if w["flops"] <= 0.9 * biggest and w["bytes"] <= 4e9:
            return case


# ---- what a program has in hand before the call ------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _scale_dtype(case):
    return L.SCALE_FP16 if case["scales"] == "fp16" else L.SCALE_BF16


def prepare(case, seed):
    if case["kind"] == "gemv":
        M, K, T = case["rows"], case["cols"], case["tokens"]
        g = _gen(seed)
        sdt = torch.float16 if case["scales"] == "fp16" else torch.bfloat16
        packed = torch.randint(0, 256, (M, K // 2), dtype=torch.uint8, device=DEV, generator=g)
        scales = (torch.randn(M, K // 128, device=DEV, generator=g).abs() * 0.02).to(sdt)
        x = torch.randn(T, K, device=DEV, generator=g).to(torch.bfloat16)
        return dict(case=case, packed=packed, scales=scales, x=x,
                    q=torch.empty(T, K, dtype=torch.int8, device=DEV),
                    sq=torch.empty(T, K // 128, device=DEV), y=torch.empty(T, M, device=DEV))
    cfg = MoeConfig("case", case["hidden"], case["experts"], case["top_k"], case["inter"],
                    case["shared"], (case["tokens"],), zipf=case["zipf"], layers=case["layers"],
                    shared_gate=case["gate"], seed=seed)
    precision = L.PRECISION_W4A8 if case["precision"] == "w4a8" else L.PRECISION_W4A16
    layers = [MoeLayer(cfg, layer=i, scale_dtype=_scale_dtype(case), precision=precision)
              for i in range(case["layers"])]
    T, H = case["tokens"], case["hidden"]
    mode = L.NORM_ONE_PLUS if case["norm"] == "one_plus" else L.NORM_PLAIN
    g = _gen(seed)
    norms = []
    for _ in layers:
        w = 0.1 * torch.randn(H, device=DEV, generator=g)
        norms.append((w if mode == L.NORM_ONE_PLUS else 1.0 + w).to(torch.bfloat16))
    st = dict(case=case, layers=layers, norms=norms, mode=mode, x=make_input(cfg, T),
              y=torch.empty(T, H, dtype=torch.bfloat16, device=DEV))
    if case["kind"] == "stack":
        st["stack"] = MoeStack(layers, norms)
        st["ws"] = st["stack"].workspace(T)
    else:
        st["ws"] = layers[0].workspace(T)
    return st


def run(st):
    kind = st["case"]["kind"]
    if kind == "gemv":
        M, K, T = st["case"]["rows"], st["case"]["cols"], st["case"]["tokens"]
        lib, stream = L.lib(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
        x, q, sq, y = (C.c_void_p(st[n].data_ptr()) for n in ("x", "q", "sq", "y"))
        L.check(lib.ainfer_moe_act_quant_i8(x, L.ACT_BF16, T, K, q, sq, stream))
        L.check(lib.ainfer_moe_int4_gemv_i8(
            C.c_void_p(st["packed"].data_ptr()), C.c_void_p(st["scales"].data_ptr()),
            _scale_dtype(st["case"]), q, sq, M, K, T, y, stream))
        return {"q": st["q"], "sq": st["sq"], "y": st["y"]}
    if kind == "stack":
        st["stack"].forward(st["x"], st["y"], st["ws"], norm_mode=st["mode"], eps=EPS)
    elif kind == "block":
        st["layers"][0].block_forward(st["x"], st["y"], st["ws"], norm_w=st["norms"][0],
                                      norm_mode=st["mode"], eps=EPS)
    else:
        st["layers"][0].forward(st["x"], st["y"], st["ws"])
    return st["y"]


# ---- what a pass cannot do without -------------------------------------------
def _experts_hit(case):
    """Distinct routed experts of one step, expected (router logits of normal
    inputs are normal; a Zipf bias is simulated once on fixed numbers)."""
    E, k, T = case["experts"], case["top_k"], case["tokens"]
    if case["zipf"] == 0.0:
        return E * (1.0 - (1.0 - k / E) ** T)
    T = min(T, 4096)
    r = np.random.default_rng(1)
    logits = (r.standard_normal((T, E)) * 0.02 * math.sqrt(case["hidden"])
              - case["zipf"] * np.log(np.arange(1, E + 1)))
    return float(np.unique(np.argpartition(-logits, k - 1, axis=1)[:, :k]).size)


def work(case):
    T = case["tokens"]
    if case["kind"] == "gemv":
        M, K = case["rows"], case["cols"]
        return {"bytes": M * K // 2 + M * K // 128 * 2 + T * K * 2 + T * K + T * K // 128 * 4
                + T * M * 4, "flops": 2 * T * M * K}
    H, E, k, I, Is = (case[n] for n in ("hidden", "experts", "top_k", "inter", "shared"))
    expert = 3 * H * I // 2 + 3 * H * I // 128 * 2
    shared = 3 * H * Is // 2 + 3 * H * Is // 128 * 2
    layer = _experts_hit(case) * expert + shared + E * H * 2 + H * 2
    n = case["layers"]
    return {"bytes": int(n * layer + 2 * T * H * 2),
            "flops": n * (2 * T * 3 * H * (k * I + Is) + 2 * T * H * E)}


def tolerance(case):
    # each is about four times what a summation in another order, or the 64-bit
    # results, were measured to differ by
    if case["kind"] == "gemv":  # 32-bit sums of exact integer dots
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    if case["kind"] == "stack":  # a bf16 residual stream through several layers
        return {"rel": 3e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.1}


# ---- the same in 64 bits -----------------------------------------------------
def _f64(packed, scales, rows, K):
    """[rows][K] float64 of packed int4 (low nibble = even k) with one scale per 128."""
    p = packed.view(rows, K // 2)
    q = torch.stack((p & 15, p >> 4), dim=-1).view(rows, K).to(torch.int8)
    q = torch.where(q > 7, q - 16, q)
    s = scales.view(rows, K // 128).double()
    return (q.view(rows, K // 128, 128).double() * s.unsqueeze(-1)).view(rows, K)


def _quantized(x):
    """The int8 form of x per group of 128 (codes and scales as the format
    defines them: from 32-bit values), back in 64 bits."""
    g = x.float().view(x.shape[0], -1, 128)
    top = g.abs().amax(-1, keepdim=True)
    s = top / torch.full_like(top, 127.0)  # a true division: by a constant it may be a product
    s = torch.where(s == 0, torch.ones_like(s), s)
    r = g / s
    c = torch.trunc(torch.where(r >= 0, r + 0.5, r - 0.5)).clamp(-127, 127)
    return (c.double() * s.double()).view(x.shape)


def _mlp(x, t, pre, e, H, I, w4a8):
    def mat(name, rows, K):
        w, s = t[pre[0] + name], t[pre[1] + name]
        nb, ns = rows * K // 2, rows * K // 128
        return _f64(w[e * nb:(e + 1) * nb], s[e * ns:(e + 1) * ns], rows, K)

    g, u = x @ mat("gate", I, H).t(), x @ mat("up", I, H).t()
    a = g / (1.0 + torch.exp(-g)) * u
    return (_quantized(a) if w4a8 else a) @ mat("down", H, I).t()


def _layer64(case, ly, x):
    """The layer on the bf16 rows x, in 64 bits."""
    H, E, k, I, Is = (case[n] for n in ("hidden", "experts", "top_k", "inter", "shared"))
    t, w4a8 = ly.t, case["precision"] == "w4a8"
    xd = x.double()
    logits = xd @ t["router_w"].view(E, H).double().t()
    if t["router_bias"] is not None:
        logits = logits + t["router_bias"].double()
    val, idx = torch.sort(logits, dim=1, descending=True, stable=True)
    idx, w = idx[:, :k], torch.softmax(val[:, :k], dim=1)
    xin = _quantized(x) if w4a8 else xd
    y = torch.zeros_like(xd)
    for e in torch.unique(idx).tolist():
        tok, slot = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, tok, _mlp(xin[tok], t, ("w_", "s_"), e, H, I, w4a8)
                     * w[tok, slot].unsqueeze(1))
    if Is:
        s = _mlp(xin, t, ("ws_", "ss_"), 0, H, Is, w4a8)
        if t["shared_gate_w"] is not None:
            s = s * torch.sigmoid(xd @ t["shared_gate_w"].double()).unsqueeze(1)
        y = y + s
    return y


def exact(case, seed):
    st = prepare(case, seed)
    if case["kind"] == "gemv":
        w = _f64(st["packed"], st["scales"], case["rows"], case["cols"])
        return {"q": None, "sq": st["x"].double().view(case["tokens"], -1, 128).abs().amax(-1) / 127,
                "y": _quantized(st["x"]) @ w.t()}
    if case["kind"] == "forward":
        return _layer64(case, st["layers"][0], st["x"])
    # the residual stream and the normalized rows are bf16 by definition; the
    # last sum stays in 64 bits
    r = st["x"].double()
    for i, (ly, nw) in enumerate(zip(st["layers"], st["norms"])):
        if i:
            r = r.to(torch.bfloat16).double()
        w = nw.double() + (1.0 if case["norm"] == "one_plus" else 0.0)
        h = r / torch.sqrt((r * r).mean(1, keepdim=True) + EPS) * w
        r = r + _layer64(case, ly, h.to(torch.bfloat16))
    return r
