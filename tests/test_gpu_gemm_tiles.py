"""The prefill expert GEMM at the edges of its tiles: experts of 1 to 300
tokens (every 16-token subtile count; tiles of at most 16, 32 and 64 tokens,
which the shapes below take), K of 1, 2, 5, 11, 15, 18 and 32 quantization
groups (odd and even), rows that do not fill a block.

Each expert row is compared with the float64 MLP of the dequantised weights.
The bound per element is what the arithmetic states: fp32 sums of n exact
products (n * 2^-24 of the sum of magnitudes), the activation rounded to bf16 (8
significant bits: half a unit in the last place is at most 2^-8 of the value;
and 2^-20 for the exp2 / rcp SiLU), the output rounded to bf16 (2^-8).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


COUNTS = {"low": [1, 15, 16, 17, 31, 32, 33, 47, 48, 60], "high": [49, 63, 64, 65, 59]}
T = 300


def routing(counts):
    """Slot 0: expert i gets counts[i] tokens, scattered; slot 1: expert E - 1 all of them."""
    rng = np.random.default_rng(5)
    first = np.repeat(np.arange(len(counts)), counts)
    assert first.size == T
    rng.shuffle(first)
    return first


@pytest.mark.parametrize("scales", ["fp16", "bf16"])
@pytest.mark.parametrize("which", ["low", "high"])
@pytest.mark.parametrize("H,I,Is", [(4096, 128, 128), (2304, 256, 128), (1920, 1408, 0),
                                    (128, 128, 1920), (640, 2304, 256), (4096, 2304, 256)])
def test_expert_rows_at_tile_edges(torch, oracle, H, I, Is, which, scales):
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    print(f"[case] gemm tiles H={H} I={I} Is={Is} {which} {scales}", flush=True)
    E = 12
    cfg = MoeConfig("tiles", H, E, 2, I, Is, (T,), seed=77)
    sd = L.SCALE_FP16 if scales == "fp16" else L.SCALE_BF16
    ly = MoeLayer(cfg, scale_dtype=sd)
    first = routing(COUNTS[which])
    idx = np.stack([first, np.full(T, E - 1)], 1).astype(np.int32)
    x = make_input(cfg, T)
    o = ly.experts(x, torch.from_numpy(idx).cuda(), ly.workspace(T))
    torch.cuda.synchronize()
    got = o.double().cpu()
    xd = x.double().cpu()

    def mat(pre, name, e, rows, K):
        w = ly.t[pre[0] + name].cpu().numpy().reshape(-1, rows, K // 2)[e]
        s = ly.t[pre[1] + name].view(torch.int16).cpu().numpy().view(np.uint16)
        w = oracle.dequant(w, s.reshape(-1, rows, K // 128)[e], sd, rows, K)
        return torch.from_numpy(np.asarray(w, np.float64).reshape(rows, K))

    def check(rows, tok, pre, e, inter):
        g, u, d = mat(pre, "gate", e, inter, H), mat(pre, "up", e, inter, H), mat(pre, "down", e, H, inter)
        xi = xd[tok]
        vg, vu = xi @ g.t(), xi @ u.t()
        eps = 2.0 ** -24
        dg, du = (H + 300) * eps * (xi.abs() @ g.abs().t()), (H + 300) * eps * (xi.abs() @ u.abs().t())
        sil = vg / (1 + torch.exp(-vg))
        act = sil * vu
        # |silu'| <= 1.1
        dact = 1.1 * dg * (vu.abs() + du) + sil.abs() * du + act.abs() * (2.0 ** -8 + 2.0 ** -20)
        ref = act @ d.t()
        mag = (act.abs() + dact) @ d.abs().t()
        bound = dact @ d.abs().t() + (inter + 300) * eps * mag
        bound = bound + 2.0 ** -8 * (ref.abs() + bound) + 1e-30
        err = (got[rows] - ref).abs()
        worst = float((err / bound).max())
        assert worst <= 1.0, (e, len(tok), worst)

    for e in range(len(COUNTS[which])):
        tok = np.nonzero(first == e)[0]
        check(tok * 2, tok, ("w_", "s_"), e, I)
    every = np.arange(T)
    check(every * 2 + 1, every, ("w_", "s_"), E - 1, I)
    if Is:
        check(2 * T + every, every, ("ws_", "ss_"), 0, Is)


# (H, E, k, I, Is) and the token counts either side of the rule that sends the
# experts to the GEMM: 3.25 tokens per expert, and up to about 20 where the
# stages have few items
EDGES = [((1024, 64, 8, 256, 256), (25, 26, 64, 65)),
         ((512, 8, 2, 256, 384), (47, 48, 65)),
         ((3584, 20, 4, 128, 0), (24, 25, 111, 112)),
         ((640, 130, 3, 128, 0), (140, 141))]


@pytest.mark.parametrize("dims,T", [(d, t) for d, ts in EDGES for t in ts])
def test_forward_either_side_of_the_gemm_rule(torch, oracle, dims, T):
    """The whole layer on both sides of the rule, in the fused (T <= 64) and
    the staged dispatch, against the oracle, and its stages composed against
    it (the stage entry takes the same rule)."""
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    print(f"[case] gemm rule {dims} T={T}", flush=True)
    H, E, k, I, Is = dims
    cfg = MoeConfig("rule", H, E, k, I, Is, (T,), seed=3)
    ly = MoeLayer(cfg)
    x = make_input(cfg, T)
    ws = ly.workspace(T)
    y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device="cuda")
    ly.forward(x, y, ws)
    idx, w, sg, _ = ly.route(x, ws)
    y2 = torch.empty_like(y)
    ly.combine(ly.experts(x, idx, ws), w, sg, y2)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))

    def bits(t):
        return (t.view(torch.int16) if t.dtype in (torch.bfloat16, torch.float16) else t).cpu().numpy()

    host = oracle.HostLayer(cfg.shape_tuple(), {
        n: None if t is None else bits(t).view(np.uint16) if t.dtype in (torch.bfloat16, torch.float16)
        else bits(t) for n, t in ly.t.items()}, ly.shape.scale_dtype)
    ref = host.forward(bits(x).view(np.uint16), T).astype(np.float64)
    got = y.double().cpu().numpy()
    assert np.abs(got - ref).max() <= 2e-2 * np.abs(ref).max()  # the layer's bf16 tolerance


@pytest.mark.parametrize("scales", ["fp16", "bf16"])
@pytest.mark.parametrize("H,E,k,I,Is", [(4096, 6, 2, 128, 128), (2304, 24, 3, 256, 1280),
                                        (1920, 3, 1, 896, 0), (128, 5, 5, 128, 1920),
                                        (1024, 64, 8, 384, 256), (1920, 12, 2, 1408, 0),
                                        (640, 12, 2, 2304, 256)])
def test_w4a8_gemm_gives_the_decode_rows(torch, H, E, k, I, Is, scales):
    """In W4A8 a token's output does not depend on how many tokens share the
    call: every product and sum is defined by the format, so the GEMM's rows
    (T > 16: tiles of 1 to 64 tokens, fused, staged and counted dispatch)
    equal, bit for bit, the decode kernels' rows of the same tokens in calls
    of 16."""
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    sd = L.SCALE_FP16 if scales == "fp16" else L.SCALE_BF16
    cfg = MoeConfig("w8tiles", H, E, k, I, Is, (T,), seed=78)
    ly = MoeLayer(cfg, scale_dtype=sd, precision=L.PRECISION_W4A8)
    x = make_input(cfg, T) * 2
    x[3] = 0  # a group of zeros has scale 1
    ws = ly.workspace(T)
    want = torch.empty_like(x)
    for t in range(0, T, 16):
        ly.forward(x[t:t + 16], want[t:t + 16], ws)
    for n in (17, 33, 64, 65, 150, T):
        print(f"[case] w4a8 gemm H={H} E={E} I={I} Is={Is} {scales} T={n}", flush=True)
        y = torch.full((n, H), float("nan"), dtype=torch.bfloat16, device="cuda")
        ly.forward(x[:n], y, ws)
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want[:n].view(torch.int16)), n


@pytest.mark.parametrize("H,E,T", [(128, 96, 257), (256, 512, 511), (256, 512, 1025), (128, 512, 2048),
                                   (384, 500, 2049), (2560, 64, 300), (4096, 40, 256),
                                   (1152, 513, 1025), (2048, 1024, 1030)])
def test_router_at_tile_edges(torch, oracle, H, E, T):
    """The prefill router at the edges of its GEMM tiles (32 x 64, 64 x 64, 64 x
    128 of tokens x experts, the first and last count of items of each; K of 2
    to 64 steps): the selection is canonical, so indices are the oracle's, and
    the weights and gate differ by expf (an ulp on each side), the sum of 6 and a
    division: below 16 ulps, 2^-19.  Columns with
    one bias and equal experts make ties, which the smaller index wins."""
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    from test_gpu_parity import host_copy, to_np
    print(f"[case] router tiles H={H} E={E} T={T}", flush=True)
    cfg = MoeConfig("rt", H, E, 6, 128, 128, (T,), seed=5)
    ly = MoeLayer(cfg)
    rw = ly.t["router_w"].view(E, H)
    rw[1::7] = rw[0]
    x = make_input(cfg, T)
    idx, w, sg, _ = ly.route(x, ly.workspace(T))
    torch.cuda.synchronize()
    r_idx, r_w, r_sg, _ = host_copy(oracle, ly).route(to_np(x), T)
    assert np.array_equal(idx.cpu().numpy(), r_idx)
    np.testing.assert_allclose(w.cpu().numpy(), r_w, rtol=2.0 ** -19, atol=0)
    np.testing.assert_allclose(sg.cpu().numpy(), r_sg, rtol=2.0 ** -19, atol=0)


@pytest.mark.parametrize("T", [33, 300, 1100])
def test_router_rows_without_a_threshold(torch, oracle, T):
    """A token whose logits are NaN or infinite has no candidate threshold: its
    experts are still k distinct valid ones, and every other row is the oracle's."""
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    from test_gpu_parity import host_copy, to_np
    print(f"[case] router non-finite rows T={T}", flush=True)
    E, k = 96, 6
    cfg = MoeConfig("rn", 512, E, k, 128, 128, (T,), seed=6)
    ly = MoeLayer(cfg)
    x = make_input(cfg, T)
    bad = [5, T - 1]
    good = np.setdiff1d(np.arange(T), bad)
    r_idx, _, _, _ = host_copy(oracle, ly).route(to_np(x), T)
    x[5] = float("nan")
    x[T - 1, 7] = float("inf")
    idx, _, _, _ = ly.route(x, ly.workspace(T))
    torch.cuda.synchronize()
    idx = idx.cpu().numpy()
    assert np.array_equal(idx[good], r_idx[good])
    for t in bad:
        assert idx[t].min() >= 0 and idx[t].max() < E and np.unique(idx[t]).size == k
