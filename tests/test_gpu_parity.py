"""HIP path vs the CPU oracle on the same seeded inputs, through the C ABI.

Bars: router logits, top-k indices and the dispatch permutation bit-exact;
layer outputs max|y - ref| / max|ref| <= 2e-2 and cosine >= 0.9999 (the
bf16 tolerance of the benchmark definition); RMSNorm bit-exact.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_TOL = 2e-2
COS_MIN = 0.9999


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def to_np(t):
    import torch
    if t.dtype in (torch.bfloat16, torch.float16):
        return t.view(torch.int16).cpu().numpy().view(np.uint16)
    return t.cpu().numpy()


def host_copy(oracle, layer):
    arrays = {n: (to_np(t) if t is not None else None) for n, t in layer.t.items()}
    return oracle.HostLayer(layer.cfg.shape_tuple(), arrays, layer.shape.scale_dtype)


def check_close(y_bf16, ref, what=""):
    y = (y_bf16.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    ref = ref.astype(np.float64)
    rel = np.abs(y - ref).max() / np.abs(ref).max()
    cos = float((y * ref).sum() / np.sqrt((y * y).sum() * (ref * ref).sum()))
    print(f"[parity] {what} rel={rel:.3e} cos={cos:.7f}", flush=True)
    assert rel <= REL_TOL, (what, rel)
    assert cos >= COS_MIN, (what, cos)
    return rel, cos


_layers = {}


def get_layer(torch, name, **over):
    from ainfer_amd.moe import MoeLayer
    from ainfer_amd.synthetic import CONFIGS
    import dataclasses
    key = (name, tuple(sorted(over.items())))
    if key not in _layers:
        cfg = dataclasses.replace(CONFIGS[name], **over) if over else CONFIGS[name]
        _layers.clear()            # keep one layer resident at a time
        torch.cuda.empty_cache()
        _layers[key] = MoeLayer(cfg)
        torch.cuda.synchronize()
    return _layers[key]


def test_fill_matches_oracle(torch, oracle):
    layer = get_layer(torch, "c0")
    want = oracle.HostLayer.synthetic(layer.cfg)
    got = host_copy(oracle, layer)
    for n, a in want.a.items():
        if a is None:
            assert got.a[n] is None
            continue
        assert np.array_equal(got.a[n].view(a.dtype) if a.dtype != np.float32 else got.a[n], a), n


# T = 5 and 8: two tokens per wave in 8-wave routing workgroups; 16: 16-wave workgroups
ROUTE_CASES = [("c0", 1), ("c1", 1), ("c1", 4), ("c1", 5), ("c1", 8), ("c1", 16), ("c3", 8), ("c3", 64),
               ("c2", 4096)]


@pytest.mark.parametrize("name,T", ROUTE_CASES)
def test_route_and_dispatch_bit_exact(torch, oracle, name, T):
    from ainfer_amd.moe import make_input
    print(f"[case] route {name} T={T}", flush=True)
    layer = get_layer(torch, name)
    x = make_input(layer.cfg, T, tag=T)
    ws = layer.workspace(T)
    idx, w, sg, lg = layer.route(x, ws, want_logits=True)
    counts, offsets, perm, inv = layer.dispatch(idx, ws)
    torch.cuda.synchronize()
    hl = host_copy(oracle, layer)
    xh = to_np(x)
    r_idx, r_w, r_sg, r_lg = hl.route(xh, T)
    assert np.array_equal(to_np(lg).view(np.uint32), r_lg.view(np.uint32)), "logits"
    _report_topk_mismatch(to_np(idx), r_idx, r_lg)
    assert np.array_equal(to_np(idx), r_idx), "top-k indices"
    np.testing.assert_allclose(to_np(w), r_w, rtol=2e-6, atol=1e-7)
    np.testing.assert_allclose(to_np(sg), r_sg, rtol=2e-6, atol=1e-7)
    c, o, p, iv = oracle.dispatch(r_idx, layer.cfg.n_experts)
    assert np.array_equal(to_np(counts), c)
    assert np.array_equal(to_np(offsets), o)
    assert np.array_equal(to_np(perm), p), "dispatch permutation"
    assert np.array_equal(to_np(inv), iv)


def _report_topk_mismatch(got, want, logits):
    """Print the rows whose top-k differs (indices and the logits of every
    expert either side picked) before the assertion fails."""
    bad = np.where((got != want).any(axis=1))[0]
    if len(bad):
        print(f"[topk] {len(bad)} rows differ: {bad[:16].tolist()}", flush=True)
        for t in bad[:4]:
            es = sorted(set(got[t].tolist()) | set(want[t].tolist()))
            print(f"[topk] t={t} got={got[t].tolist()} want={want[t].tolist()} "
                  f"logits={[(e, float(logits[t, e])) for e in es]}", flush=True)


def _route_check(torch, oracle, layer, x, what):
    T = x.shape[0]
    ws = layer.workspace(T)
    idx, w, sg, lg = layer.route(x, ws, want_logits=True)
    torch.cuda.synchronize()
    hl = host_copy(oracle, layer)
    r_idx, r_w, r_sg, r_lg = hl.route(to_np(x), T)
    assert np.array_equal(to_np(lg).view(np.uint32), r_lg.view(np.uint32)), what
    assert np.array_equal(to_np(idx), r_idx), what
    np.testing.assert_allclose(to_np(w), r_w, rtol=2e-6, atol=1e-7)
    return r_idx


def test_router_ties_and_degenerate_inputs(torch, oracle):
    """Inputs built to defeat the candidate refine: exact ties (duplicated
    router rows), all logits equal (every expert a candidate), coarse values
    with many near and exact ties, and large-magnitude activations."""
    from ainfer_amd.moe import make_input
    layer = get_layer(torch, "c1")
    E, H = layer.cfg.n_experts, layer.cfg.hidden
    rw0 = layer.t["router_w"].clone()
    for T in (1, 16, 64, 300):
        x = make_input(layer.cfg, T, tag=77 + T)
        # duplicated rows: experts 2i and 2i+1 always tie
        rw = rw0.view(E, H).clone()
        rw[1::2] = rw[0::2]
        layer.set_tensor("router_w", rw.reshape(-1).contiguous())
        idx = _route_check(torch, oracle, layer, x, f"dup rows T={T}")
        assert (idx[:, ::2] % 2 == 0).all()  # lower index of each tied pair first
        # all logits equal: top-k is experts 0..k-1
        layer.set_tensor("router_w", torch.zeros_like(rw0))
        idx = _route_check(torch, oracle, layer, x, f"zeros T={T}")
        assert (idx == np.arange(layer.cfg.top_k)).all()
        # coarse values: many exact and near ties
        q = torch.randint(-1, 2, rw0.shape, device="cuda").to(torch.bfloat16) * 0.015625
        xq = torch.randint(-2, 3, x.shape, device="cuda").to(torch.bfloat16)
        layer.set_tensor("router_w", q.contiguous())
        _route_check(torch, oracle, layer, xq, f"coarse T={T}")
        # large activations
        layer.set_tensor("router_w", rw0)
        _route_check(torch, oracle, layer, (x.float() * 4096).to(torch.bfloat16), f"big T={T}")
    layer.set_tensor("router_w", rw0)


FWD_CASES = [("c0", 1), ("c1", 1), ("c1", 2), ("c1", 4), ("c1", 16), ("c1", 100), ("c3", 1), ("c3", 64)]


@pytest.mark.parametrize("name,T", FWD_CASES)
def test_forward_parity(torch, oracle, name, T):
    from ainfer_amd.moe import make_input
    print(f"[case] forward {name} T={T}", flush=True)
    layer = get_layer(torch, name)
    x = make_input(layer.cfg, T, tag=100 + T)
    ws = layer.workspace(T)
    y = torch.full((T, layer.cfg.hidden), float("nan"), dtype=torch.bfloat16, device="cuda")
    layer.forward(x, y, ws)
    torch.cuda.synchronize()
    assert not torch.isnan(y).any(), "kernel left poisoned outputs"
    ref = host_copy(oracle, layer).forward(to_np(x), T)
    check_close(to_np(y), ref, f"{name} T={T}")
    # bitwise run-to-run determinism
    y2 = torch.empty_like(y)
    layer.forward(x, y2, ws)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))


def test_decode_sync_words_return_to_zero(torch, oracle):
    """Every decode call leaves the workspace's counters and logit slots zero
    and no bounded wait runs out, over all decode token counts in a row."""
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import make_input
    layer = get_layer(torch, "c1")
    ws = layer.workspace(16)
    assert layer.workspace_check(ws) == L.OK
    y = torch.empty(16, layer.cfg.hidden, dtype=torch.bfloat16, device="cuda")
    for rep in range(3):
        for T in range(1, 17):
            layer.forward(make_input(layer.cfg, T, tag=200 + T), y[:T], ws)
    rc = layer.workspace_check(ws)
    assert rc == L.OK, L.lib().ainfer_moe_strerror(rc).decode()
    # the route-only entry shares the logit slots
    x = make_input(layer.cfg, 16, tag=9)
    layer.route(x, ws, want_logits=True)
    assert layer.workspace_check(ws) == L.OK


def test_prefill_zipf_parity_on_token_sample(torch, oracle):
    """c2 at full size (T = 4096): tokens are independent given routing, so
    the oracle recomputes a sample of rows; the whole output is checked for
    determinism and finiteness."""
    from ainfer_amd.moe import make_input
    T = 4096
    print(f"[case] forward c2 T={T}", flush=True)
    layer = get_layer(torch, "c2")
    x = make_input(layer.cfg, T, tag=7)
    ws = layer.workspace(T)
    y = torch.full((T, layer.cfg.hidden), float("nan"), dtype=torch.bfloat16, device="cuda")
    layer.forward(x, y, ws)
    torch.cuda.synchronize()
    assert torch.isfinite(y.float()).all()
    rng = np.random.default_rng(0)
    rows = np.sort(rng.choice(T, size=96, replace=False))
    rows[0], rows[-1] = 0, T - 1
    xh = to_np(x)[rows]
    ref = host_copy(oracle, layer).forward(np.ascontiguousarray(xh), len(rows))
    check_close(to_np(y)[rows], ref, "c2 T=4096 sample")
    y2 = torch.empty_like(y)
    layer.forward(x, y2, ws)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))


def midpoint_row(H, torch, tiny=True):
    """A row (H = 2048 or 4096) whose mean square is a float midpoint,
    0.5 + 2^-25: H/2 ones and H/2048 elements 2^-7.  Its sum of squares is
    exact in every order, so the device takes the tree sum (exactness test).
    With `tiny`, one element 2^-40 makes the sum inexact while the mean stays
    within 2^-70 of the midpoint: neither test passes and the RMSNorm takes
    its sequential re-sum."""
    r = torch.zeros(H, dtype=torch.float32)
    r[:H // 2] = 1.0
    r[H // 2:H // 2 + H // 2048] = 2.0 ** -7
    if tiny:
        r[H - 3] = 2.0 ** -40
    return r.to(torch.bfloat16)


def test_rmsnorm_bit_exact(torch, oracle):
    """Against the oracle, which sums as the reference does (sequentially for
    H != 5120, kernels.cpp:86-97; as the 256-lane tree at 5120)."""
    from ainfer_amd.moe import rmsnorm
    from ainfer_amd import _lib as L
    for T, H in ((1, 4096), (8, 2048), (3, 1000), (4, 5120), (64, 4096)):
        x = torch.randn(T, H, device="cuda").to(torch.bfloat16) * 3
        if H == 4096 or H == 2048:
            x[0] = midpoint_row(H, torch).cuda()
            if T > 2:
                x[1] = midpoint_row(H, torch, tiny=False).cuda()
                x[2, 7] = 2.0 ** -50      # inexact sum: the interval test
        w = torch.randn(H, device="cuda").to(torch.bfloat16)
        for mode in (L.NORM_PLAIN, L.NORM_ONE_PLUS):
            for ww in (None, w):
                y = torch.empty_like(x)
                rmsnorm(x, y, ww, mode)
                torch.cuda.synchronize()
                ref = oracle.rmsnorm_bf16(to_np(x), None if ww is None else to_np(ww), mode)
                assert np.array_equal(to_np(y), ref), (T, H, mode, ww is None)


def test_block_forward_and_stack(torch, oracle):
    """Three chained blocks (RMSNorm -> MoE -> residual) of the c3/c4 layer
    shape with 64 experts, bf16 residual carried between them."""
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import CONFIGS
    import dataclasses
    cfg = dataclasses.replace(CONFIGS["c4"], n_experts=64, layers=3)
    T = 8
    _layers.clear()
    layers = [MoeLayer(cfg, layer=i) for i in range(3)]
    r = make_input(cfg, T, tag=3) * 4
    ws = layers[0].workspace(T)
    r_gpu = r.clone()
    hls = [host_copy(oracle, L) for L in layers]
    r_ref = to_np(r)
    for i, L in enumerate(layers):
        # per block: same input on both sides, so top-k after RMSNorm is exact
        inp = r_gpu.clone()
        L.block_forward(inp, r_gpu, ws)
        torch.cuda.synchronize()
        want = hls[i].block_forward(to_np(inp), T)
        h = oracle.rmsnorm_bf16(to_np(inp), None, oracle.NORM_PLAIN)
        idx, *_ = L.route(torch.from_numpy(h.view(np.int16)).view(torch.bfloat16).cuda(), ws)
        r_idx, *_ = hls[i].route(h, T)
        assert np.array_equal(to_np(idx), r_idx)
        check_close(to_np(r_gpu), oracle.bf16_to_f32(want), f"block {i}")
        r_ref = hls[i].block_forward(r_ref, T)
    # the chained CPU stack vs the chained GPU stack
    check_close(to_np(r_gpu), oracle.bf16_to_f32(r_ref), "3-block stack")


@pytest.mark.parametrize("mode", ["plain", "one_plus"])
def test_block_forward_fused_norm(torch, oracle, mode):
    """At T <= 4 the routing kernel applies the block's RMSNorm itself (one
    code path for T = 1..4).  At T = 3 to 16 every later stage is the one
    T = 17 runs (4-token tiles, per-token arithmetic), and T = 17 normalizes
    with the separate RMSNorm kernel: each token's output must be equal bit
    for bit (T = 5 and 8: both normalize with the separate kernel).  At T = 1 and 2
    down splits K differently (two k-groups to a sum), so there the check is the oracle's block within tolerance
    (as at every T)."""
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import CONFIGS
    import dataclasses
    nm = L.NORM_PLAIN if mode == "plain" else L.NORM_ONE_PLUS
    cfg = dataclasses.replace(CONFIGS["c4"], n_experts=64, layers=1)
    _layers.clear()
    layer = MoeLayer(cfg, layer=7)
    x = make_input(cfg, 17, tag=41) * 3
    x[1] = midpoint_row(cfg.hidden, torch).cuda()   # the sequential re-sum in both kernels
    x[2] = midpoint_row(cfg.hidden, torch, tiny=False).cuda()  # exact sum on a midpoint
    x[3, 11] = 2.0 ** -50                           # inexact sum: the interval test
    g = torch.Generator().manual_seed(5)
    nw = (torch.randn(cfg.hidden, generator=g) * 0.5 + (0.0 if nm == L.NORM_ONE_PLUS else 1.0))
    nw = nw.to(torch.bfloat16).cuda()
    ws = layer.workspace(17)
    ref17 = torch.empty_like(x)
    layer.block_forward(x, ref17, ws, norm_w=nw, norm_mode=nm)
    hl = host_copy(oracle, layer)
    for T in (1, 2, 3, 4, 5, 8, 16):
        print(f"[case] fused norm {mode} T={T}", flush=True)
        out = torch.empty_like(x[:T])
        layer.block_forward(x[:T].contiguous(), out, ws, norm_w=nw, norm_mode=nm)
        torch.cuda.synchronize()
        if T >= 3:
            assert torch.equal(out, ref17[:T]), f"T={T}: fused RMSNorm differs from k_rmsnorm's"
        want = hl.block_forward(to_np(x[:T].contiguous()), T, norm_w=to_np(nw), mode=nm)
        check_close(to_np(out), oracle.bf16_to_f32(want), f"fused norm T={T}")
    assert layer.workspace_check(ws) == 0


def test_zero_tokens_and_errors(torch, oracle):
    from ainfer_amd import _lib as L
    layer = get_layer(torch, "c0")
    ws = layer.workspace(4)
    x = torch.zeros(0, layer.cfg.hidden, dtype=torch.bfloat16, device="cuda")
    layer.forward(x, x, ws)
    x = torch.zeros(8, layer.cfg.hidden, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(L.MoeError):
        layer.forward(x, x.clone(), ws)       # workspace sized for 4 tokens


@pytest.mark.parametrize("name,T", [("c1", 1), ("c1", 16), ("c1", 300), ("c3", 64)])
def test_forward_parity_bf16_scales(torch, oracle, name, T):
    """The reference's own scale dtype (bf16, binfer.py:76-91) through every
    expert path: down with the combine in it (T=1), the streaming items
    (T=16, and c3 T=64) and the grouped GEMM (T=300)."""
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import CONFIGS
    print(f"[case] forward bf16 scales {name} T={T}", flush=True)
    _layers.clear()
    torch.cuda.empty_cache()
    layer = MoeLayer(CONFIGS[name], scale_dtype=L.SCALE_BF16)
    x = make_input(layer.cfg, T, tag=500 + T)
    ws = layer.workspace(T)
    y = torch.full((T, layer.cfg.hidden), float("nan"), dtype=torch.bfloat16, device="cuda")
    layer.forward(x, y, ws)
    torch.cuda.synchronize()
    assert not torch.isnan(y).any()
    ref = host_copy(oracle, layer).forward(to_np(x), T)
    check_close(to_np(y), ref, f"bf16 scales {name} T={T}")
    del layer


# shapes at the validation limits: E = 1024 experts, k = 32 (above the fast
# top-k's 16), no shared expert; H = I = 128 (one k-group); H = I = 4096
EDGE = {
    "wide": dict(hidden=1024, n_experts=1024, top_k=32, inter=128, shared_inter=0),
    "narrow": dict(hidden=128, n_experts=8, top_k=8, inter=128, shared_inter=128),
    "deep": dict(hidden=4096, n_experts=16, top_k=2, inter=4096, shared_inter=4096),
}


EDGE_CASES = [(e, T) for e in ("wide", "narrow") for T in (1, 5, 16, 40, 300)] + \
    [("deep", T) for T in (1, 5, 16, 40)]


@pytest.mark.parametrize("edge,T", EDGE_CASES)
def test_forward_parity_at_shape_limits(torch, oracle, edge, T):
    """Route (bit-exact top-k and permutation) and forward parity on shapes
    at the validation limits, through every T regime (decode kernels,
    16-token tiles, prefill GEMM)."""
    import dataclasses
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import CONFIGS
    print(f"[case] edge {edge} T={T}", flush=True)
    cfg = dataclasses.replace(CONFIGS["c1"], name=f"edge_{edge}", **EDGE[edge])
    _layers.clear()
    torch.cuda.empty_cache()
    layer = MoeLayer(cfg)
    x = make_input(cfg, T, tag=900 + T)
    ws = layer.workspace(T)
    hl = host_copy(oracle, layer)
    idx, w, sg, lg = layer.route(x, ws, want_logits=True)
    torch.cuda.synchronize()
    r_idx, r_w, r_sg, r_lg = hl.route(to_np(x), T)
    assert np.array_equal(to_np(lg).view(np.uint32), r_lg.view(np.uint32)), "logits"
    assert np.array_equal(to_np(idx), r_idx), "top-k"
    y = torch.full((T, cfg.hidden), float("nan"), dtype=torch.bfloat16, device="cuda")
    layer.forward(x, y, ws)
    torch.cuda.synchronize()
    assert not torch.isnan(y).any()
    check_close(to_np(y), hl.forward(to_np(x), T), f"edge {edge} T={T}")
    del layer


def _random_shapes(n, seed=2024):
    rng = np.random.default_rng(seed)
    out = []
    while len(out) < n:
        H = int(rng.choice([128, 256, 384, 512, 1024, 2048]))
        E = int(rng.choice([1, 2, 3, 7, 16, 33, 64, 100, 256]))
        k = int(rng.integers(1, min(E, 12) + 1))
        I = int(rng.choice([128, 256, 384, 512]))
        Is = int(rng.choice([0, 128, 256, 512]))
        T = int(rng.choice([1, 2, 3, 7, 16, 17, 64, 65, 255, 256, 300]))
        out.append((H, E, k, I, Is, T))
    return out


@pytest.mark.parametrize("H,E,k,I,Is,T", _random_shapes(14))
def test_forward_parity_random_shapes(torch, oracle, H, E, k, I, Is, T):
    """Seeded random shapes (odd expert counts, k = E, no shared expert,
    K of one group, token counts either side of every regime boundary):
    bit-exact routing and forward parity."""
    import dataclasses
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import CONFIGS
    print(f"[case] random H={H} E={E} k={k} I={I} Is={Is} T={T}", flush=True)
    cfg = dataclasses.replace(CONFIGS["c0"], name=f"rnd_{H}_{E}_{k}_{I}_{Is}", hidden=H,
                              n_experts=E, top_k=k, inter=I, shared_inter=Is)
    _layers.clear()
    torch.cuda.empty_cache()
    layer = MoeLayer(cfg)
    x = make_input(cfg, T, tag=T + E)
    ws = layer.workspace(T)
    hl = host_copy(oracle, layer)
    idx, w, sg, lg = layer.route(x, ws, want_logits=True)
    counts, offsets, perm, inv = layer.dispatch(idx, ws)
    torch.cuda.synchronize()
    r_idx, r_w, r_sg, r_lg = hl.route(to_np(x), T)
    assert np.array_equal(to_np(lg).view(np.uint32), r_lg.view(np.uint32)), "logits"
    assert np.array_equal(to_np(idx), r_idx), "top-k"
    c, o, p, iv = oracle.dispatch(r_idx, E)
    assert np.array_equal(to_np(perm), p) and np.array_equal(to_np(counts), c)
    y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device="cuda")
    layer.forward(x, y, ws)
    torch.cuda.synchronize()
    assert not torch.isnan(y).any()
    check_close(to_np(y), hl.forward(to_np(x), T), f"random {H},{E},{k},{I},{Is} T={T}")
    assert layer.workspace_check(ws) == 0
    del layer


def _heavy_tailed(torch, T, H, seed):
    """Student-t (2 degrees of freedom: infinite variance) activations with a
    few outliers 200x the bulk per row, rounded to bf16: the inputs the
    Irwin-Hall synthetic fill never produces."""
    rng = np.random.default_rng(seed)
    x = rng.standard_t(2.0, size=(T, H)).astype(np.float32)
    for t in range(T):
        cols = rng.choice(H, size=3, replace=False)
        x[t, cols] = rng.choice([-200.0, 200.0], size=3) * np.abs(rng.standard_normal(3)) + 1.0
    return torch.from_numpy(x).to(torch.bfloat16).cuda()


@pytest.mark.parametrize("name,T", [("c1", 1), ("c1", 4), ("c1", 16), ("c1", 300), ("c3", 64)])
def test_forward_parity_heavy_tailed_activations(torch, oracle, name, T):
    """Heavy-tailed activations through every decode form and the prefill
    GEMM: routing bit-exact, outputs within the layer tolerance."""
    print(f"[case] heavy-tailed forward {name} T={T}", flush=True)
    layer = get_layer(torch, name)
    x = _heavy_tailed(torch, T, layer.cfg.hidden, 1000 + T)
    _route_check(torch, oracle, layer, x, f"heavy {name} T={T}")
    ws = layer.workspace(T)
    y = torch.full((T, layer.cfg.hidden), float("nan"), dtype=torch.bfloat16, device="cuda")
    layer.forward(x, y, ws)
    torch.cuda.synchronize()
    assert not torch.isnan(y).any()
    ref = host_copy(oracle, layer).forward(to_np(x), T)
    check_close(to_np(y), ref, f"heavy {name} T={T}")


def test_block_forward_heavy_tailed_residual(torch, oracle):
    """The block (RMSNorm -> layer -> residual) on a heavy-tailed residual
    stream, both the fused RMSNorm (T <= 4) and the separate kernel."""
    from ainfer_amd import _lib as L
    layer = get_layer(torch, "c1")
    ws = layer.workspace(16)
    g = torch.Generator().manual_seed(9)
    nw = (torch.randn(layer.cfg.hidden, generator=g) * 0.5 + 1.0).to(torch.bfloat16).cuda()
    hl = host_copy(oracle, layer)
    for T in (1, 4, 16):
        print(f"[case] heavy-tailed block T={T}", flush=True)
        x = _heavy_tailed(torch, T, layer.cfg.hidden, 2000 + T)
        out = torch.empty_like(x)
        layer.block_forward(x, out, ws, norm_w=nw, norm_mode=L.NORM_PLAIN)
        torch.cuda.synchronize()
        want = hl.block_forward(to_np(x), T, norm_w=to_np(nw), mode=L.NORM_PLAIN)
        check_close(to_np(out), oracle.bf16_to_f32(want), f"heavy block T={T}")
    assert layer.workspace_check(ws) == 0


@pytest.mark.parametrize("name,T", [("c1", 1), ("c1", 4), ("c1", 16), ("c1", 100), ("c1", 300),
                                    ("c3", 64)])
def test_stage_entries_compose_to_forward(torch, oracle, name, T):
    """ainfer_moe_route -> ainfer_moe_experts -> ainfer_moe_combine: within
    the layer tolerance of the oracle at every T, bit-identical to
    ainfer_moe_forward where forward runs the same expert kernels (T >= 3;
    at T <= 2 down splits K differently), and with the residual bit-identical to
    block_forward where that normalizes with the separate kernel (T > 4)."""
    from ainfer_amd.moe import make_input, rmsnorm
    print(f"[case] stage entries {name} T={T}", flush=True)
    layer = get_layer(torch, name)
    x = make_input(layer.cfg, T, tag=600 + T)
    ws = layer.workspace(T)
    idx, w, sg, _ = layer.route(x, ws)
    o = layer.experts(x, idx, ws)
    y2 = torch.empty(T, layer.cfg.hidden, dtype=torch.bfloat16, device="cuda")
    layer.combine(o, w, sg, y2)
    y = torch.empty_like(y2)
    layer.forward(x, y, ws)
    torch.cuda.synchronize()
    ref = host_copy(oracle, layer).forward(to_np(x), T)
    check_close(to_np(y2), ref, f"stages {name} T={T}")
    if T >= 3:
        assert torch.equal(y2.view(torch.int16), y.view(torch.int16)), "stages differ from forward"
    if T > 4:
        r = x * 3
        h = torch.empty_like(r)
        rmsnorm(r, h)
        idx, w, sg, _ = layer.route(h, ws)
        o = layer.experts(h, idx, ws)
        y3 = torch.empty_like(r)
        layer.combine(o, w, sg, y3, resid=r)
        yb = torch.empty_like(r)
        layer.block_forward(r, yb, ws)
        torch.cuda.synchronize()
        assert torch.equal(y3.view(torch.int16), yb.view(torch.int16)), "stages differ from block"
