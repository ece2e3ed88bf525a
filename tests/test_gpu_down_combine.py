"""The down + combine kernel of 1 to 4 tokens and the routing kernel in front of
it at every kind of shape: odd and even numbers of k-groups, experts narrower
and wider than the shared one, more tiles than waves, one expert with a long K
(its K shared by several waves), 8 and 16 rows per workgroup.

Outputs are compared with the oracle at the layer's tolerance, and bit for bit
with the stage entries, whose rows come from the item kernels: the order of
the additions is the same wherever the items' split of K is."""
import numpy as np
import pytest

from test_gpu_parity import check_close, host_copy, to_np

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


SHAPES = [(1024, 12, 5, 128, 128), (512, 9, 4, 384, 0), (640, 16, 3, 896, 1792),
          (1024, 8, 2, 768, 256), (2048, 6, 2, 1152, 0), (256, 40, 32, 256, 256),
          (384, 8, 1, 2048, 0), (512, 8, 2, 4096, 4096), (4096, 16, 6, 1024, 512),
          (4096, 12, 3, 640, 384), (128, 1, 1, 128, 128)]


@pytest.mark.parametrize("scales", ["fp16", "bf16"])
@pytest.mark.parametrize("H,E,k,I,Is", SHAPES)
def test_few_tokens_any_shape(torch, oracle, H, E, k, I, Is, scales):
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    cfg = MoeConfig("dc", H, E, k, I, Is, (4,), seed=11)
    ly = MoeLayer(cfg, scale_dtype=L.SCALE_FP16 if scales == "fp16" else L.SCALE_BF16)
    hl = host_copy(oracle, ly)
    g = torch.Generator().manual_seed(4)
    nw = (torch.randn(H, generator=g) * 0.3 + 1.0).to(torch.bfloat16).cuda()
    for T in (1, 2, 3, 4, 5):
        what = f"H={H} E={E} k={k} I={I} Is={Is} {scales} T={T}"
        print(f"[case] {what}", flush=True)
        x = make_input(cfg, T, tag=T)
        ws = ly.workspace(T)
        y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device="cuda")
        ly.forward(x, y, ws)
        idx, w, sg, lg = ly.route(x, ws, want_logits=True)
        y2 = torch.empty_like(y)
        ly.combine(ly.experts(x, idx, ws), w, sg, y2)
        b = torch.empty_like(y)
        ly.block_forward(x, b, ws, norm_w=nw)
        torch.cuda.synchronize()
        r_idx, _, _, r_lg = hl.route(to_np(x), T)
        assert np.array_equal(to_np(lg).view(np.uint32), r_lg.view(np.uint32)), what
        assert np.array_equal(to_np(idx), r_idx), what
        check_close(to_np(y), hl.forward(to_np(x), T), what)
        check_close(to_np(b), oracle.bf16_to_f32(hl.block_forward(to_np(x), T, norm_w=to_np(nw))),
                    "block " + what)
        if T >= 3 or max(I, Is) < 1024:
            assert torch.equal(y.view(torch.int16), y2.view(torch.int16)), what
        assert ly.workspace_check(ws) == 0


@pytest.mark.parametrize("H", [128, 256, 384])
def test_w4a8_block_of_a_narrow_row(torch, oracle, H):
    """The folded RMSNorm of rows with fewer 16-byte chunks than a wave has
    lanes (H < 512), in W4A8."""
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    cfg = MoeConfig("narrow", H, 16, 4, 256, 128, (4,), seed=12)
    ly = MoeLayer(cfg, precision=L.PRECISION_W4A8)
    hl = host_copy(oracle, ly)
    g = torch.Generator().manual_seed(5)
    nw = (torch.randn(H, generator=g) * 0.3 + 1.0).to(torch.bfloat16).cuda()
    for T in (1, 4):
        print(f"[case] w4a8 narrow block H={H} T={T}", flush=True)
        x = make_input(cfg, T, tag=T)
        out = torch.empty_like(x)
        ly.block_forward(x, out, ly.workspace(T), norm_w=nw)
        torch.cuda.synchronize()
        h = oracle.rmsnorm_bf16(to_np(x), to_np(nw), L.NORM_PLAIN)
        want = oracle.bf16_to_f32(to_np(x)) + hl.forward_w4a8(np.ascontiguousarray(h), T)
        check_close(to_np(out), want, f"w4a8 narrow block H={H} T={T}")


@pytest.mark.parametrize("H,E,k,I,Is", [(512, 8, 3, 128, 384), (1024, 40, 20, 512, 0),
                                        (4096, 12, 10, 1024, 256), (640, 9, 4, 896, 1792),
                                        (256, 5, 2, 2048, 128), (384, 4, 2, 2304, 256)])
def test_w4a8_rows_do_not_depend_on_the_call(torch, oracle, H, E, k, I, Is):
    """In W4A8 a token's output is defined bit by bit, so a token's row is the
    same in calls of 1, 2, 3, 4, 5 and 16 tokens, which take different kernels
    (the one-token GEMVs; the GEMM, or 16-row blocks where its items would be
    few or long; down with the combine in it up to 4 tokens), with and without
    the residual.  Against the oracle at the layer's tolerance."""
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    cfg = MoeConfig("w8dc", H, E, k, I, Is, (16,), seed=13)
    for sd in (L.SCALE_FP16, L.SCALE_BF16):
        print(f"[case] w4a8 H={H} E={E} k={k} I={I} Is={Is} scales={sd}", flush=True)
        ly = MoeLayer(cfg, scale_dtype=sd, precision=L.PRECISION_W4A8)
        x = make_input(cfg, 16, tag=3)
        ws = ly.workspace(16)
        for fn in (ly.forward, ly.block_forward):
            want, got = torch.empty_like(x), torch.empty_like(x)
            fn(x, want, ws)
            for n in (1, 2, 3, 4, 5):
                for t in range(0, 16, n):
                    fn(x[t:t + n], got[t:t + n], ws)
                torch.cuda.synchronize()
                assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (fn.__name__, n)
            if fn == ly.forward:
                check_close(to_np(want), host_copy(oracle, ly).forward_w4a8(to_np(x), 16), "w4a8 16")


@pytest.mark.parametrize("H,E,k,I,Is", [(2048, 64, 2, 1024, 0), (3584, 20, 4, 128, 128),
                                        (1024, 24, 3, 512, 256), (640, 40, 2, 384, 0),
                                        (4096, 64, 4, 512, 128)])
def test_w4a8_rows_either_side_of_the_gemm_rule(torch, H, E, k, I, Is):
    """Calls of 2 to 16 tokens go to the GEMM or to 16-row blocks by their items:
    a token's row has the same bits in all of them."""
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    print(f"[case] w4a8 rule H={H} E={E} k={k} I={I} Is={Is}", flush=True)
    cfg = MoeConfig("w8rule", H, E, k, I, Is, (17,), seed=14)
    ly = MoeLayer(cfg, precision=L.PRECISION_W4A8)
    x = make_input(cfg, 17, tag=4)
    ws = ly.workspace(17)
    want = torch.empty_like(x)
    ly.forward(x, want, ws)  # above 16 tokens: the GEMM
    for T in range(2, 17):
        y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device="cuda")
        ly.forward(x[:T], y, ws)
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want[:T].view(torch.int16)), T


@pytest.mark.parametrize("scales", ["fp16", "bf16"])
@pytest.mark.parametrize("H,E,k,I,Is", [(1024, 12, 3, 2048, 0), (512, 10, 4, 256, 1280),
                                        (1024, 6, 2, 1280, 2048), (256, 20, 16, 4096, 4096)])
def test_two_tokens_with_a_long_k(torch, oracle, H, E, k, I, Is, scales):
    """Two tokens with an expert above 1024 columns: gate/up, down and the combine
    in one launch whose workgroups meet through counters (the first three shapes;
    LDS leaves the last one three launches, and gives its T = 1 down + combine 16
    waves of 8 runs).  Every sum has the order of the one-token call's, so the
    rows are that call's bit for bit, shared experts (two tokens of one expert) and
    the residual included; calls follow each other on one workspace, whose
    counters end at zero.  Then, with every wait made to give up at once from the
    host, the outputs are NaN and the check reports it."""
    import ctypes as C
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, _ptr, _stream, make_input
    from ainfer_amd.synthetic import MoeConfig
    what = f"H={H} E={E} k={k} I={I} Is={Is} {scales} T=2"
    print(f"[case] {what}", flush=True)
    cfg = MoeConfig("two", H, E, k, I, Is, (2,), seed=15)
    ly = MoeLayer(cfg, scale_dtype=L.SCALE_FP16 if scales == "fp16" else L.SCALE_BF16)
    hl = host_copy(oracle, ly)
    ws = ly.workspace(2)
    for tag in range(4):
        x = make_input(cfg, 2, tag=tag)
        if tag == 3:
            x[1] = x[0]  # every expert has both tokens
        for fn in (ly.forward, ly.block_forward):
            y, one = torch.full_like(x, float("nan")), torch.empty_like(x)
            fn(x, y, ws)
            for t in (0, 1):
                fn(x[t:t + 1], one[t:t + 1], ws)
            torch.cuda.synchronize()
            assert torch.equal(y.view(torch.int16), one.view(torch.int16)), (what, tag, fn.__name__)
            if fn == ly.forward:
                check_close(to_np(y), hl.forward(to_np(x), 2), what)
        assert ly.workspace_check(ws) == L.OK
    try:
        L.check(L.lib().ainfer_moe_debug_spin_limit(0))
        ly.forward(x, y, ws)
        torch.cuda.synchronize()
    finally:
        L.check(L.lib().ainfer_moe_debug_spin_limit(1 << 20))
    assert torch.isnan(y.float()).all()
    assert ly.workspace_check(ws) == L.ERR_SYNC
    L.check(L.lib().ainfer_moe_workspace_init(C.byref(ly.shape), _ptr(ws), ws.numel(), _stream(None)))
    ly.block_forward(x, y, ws)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), one.view(torch.int16))
    assert ly.workspace_check(ws) == L.OK
