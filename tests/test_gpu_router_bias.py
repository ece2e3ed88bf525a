"""Router biases that are not numbers, at 1 to 17 tokens."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("bits", [-1, -2, -0x400000])  # 0xFFFFFFFF, 0xFFFFFFFE, 0xFFC00000
@pytest.mark.parametrize("dims", [(1024, 64, 6, 512, 512), (640, 65, 3, 384, 0)])
@pytest.mark.parametrize("precision", ["w4a16", "w4a8"])
def test_expert_with_a_nan_bias_is_never_selected(torch, precision, dims, bits):
    """A negative NaN sorts below every number, as -inf does, so the outputs are
    those of the layer whose bias is -inf there, bit for bit, and no wait of the
    decode routing runs out: its logit slots are their own ready flags, ~bits with
    0 for 'not yet written'."""
    from ainfer_amd import _lib as L
    from ainfer_amd.moe import MoeLayer, make_input
    from ainfer_amd.synthetic import MoeConfig
    cfg = MoeConfig("nb", *dims, (17,), zipf=1.1, seed=8)
    ly = MoeLayer(cfg, precision=L.PRECISION_W4A8 if precision == "w4a8" else L.PRECISION_W4A16)
    bias = ly.t["router_bias"]
    hot = bias.argmax().item()  # the expert that most tokens would take
    nan, ninf = bias.clone(), bias.clone()
    nan.view(torch.int32)[hot] = bits
    ninf[hot] = float("-inf")
    for T in (1, 2, 4, 5, 8, 9, 16, 17):
        print(f"[case] nan bias {bits & 0xFFFFFFFF:08x} {dims} {precision} T={T}", flush=True)
        x = make_input(cfg, T, tag=T)
        got = []
        for b in (nan, ninf):
            ly.set_tensor("router_bias", b)
            ws = ly.workspace(T)
            y, z = torch.empty_like(x), torch.empty_like(x)
            ly.forward(x, y, ws)
            ly.block_forward(x, z, ws)
            idx, w, sg, lg = ly.route(x, ws, want_logits=True)
            torch.cuda.synchronize()
            assert ly.workspace_check(ws) == 0
            assert not (idx == hot).any()
            got.append((y, z, idx, w, sg, lg))
        assert got[0][5][:, hot].isnan().all()
        assert torch.isfinite(got[0][0].float()).all()
        for a, b in zip(got[0][:5], got[1][:5]):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16)), T
