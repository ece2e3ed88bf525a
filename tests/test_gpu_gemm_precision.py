"""The fp32 steps of the prefill expert GEMM against the decode items' on the
same tokens, with weights that let each step through to the bf16 outputs."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def pack(torch, q):
    """Packed INT4 rows (low nibble = even column) of integers [..., K]."""
    q = q.to(torch.uint8) & 15
    return (q[..., 0::2] | (q[..., 1::2] << 4)).contiguous().view(-1)


def decode_rows(torch, ly, x, idx, ws):
    """The expert rows [T * k][H] of the same tokens in calls of 16."""
    k = idx.shape[1]
    return torch.cat([ly.experts(x[t:t + 16], idx[t:t + 16], ws)[:k * min(16, len(x) - t)]
                      for t in range(0, len(x), 16)])


@pytest.mark.parametrize("T,crowded", [(255, False), (255, True), (512, False)])
def test_silu_has_the_decode_items_bits(torch, T, crowded):
    """Calls below 256 tokens, and tiles of at most 32 tokens in larger ones,
    take the SiLU of the decode items (expf and a division).

    Inputs with one nonzero element and 0 / q weights make every sum exact, so
    gate and up are the same fp32 values in both, and an output is one bf16
    value silu(g) * u: the bits are equal if the SiLU's are.  Its last 16 bits
    are rounded away, hence about 400000 values: a SiLU a few units off
    changes several of them."""
    from ainfer_amd.moe import MoeLayer
    from ainfer_amd.synthetic import MoeConfig
    print(f"[case] silu bits T={T} crowded={crowded}", flush=True)
    H, E, k, I = 128, 128, (8 if T < 256 else 4), 4096
    ly = MoeLayer(MoeConfig("silu", H, E, k, I, 0, (T,), seed=21))
    g = torch.Generator(device="cuda").manual_seed(2)
    t = ly.t  # the gate's values are the random fill
    t["s_gate"].copy_(torch.rand(t["s_gate"].shape, device="cuda", generator=g) * 0.5)
    # up: row n takes column n % 128, so a token with x[j] alone has one act per
    # 128 columns; down: row h adds the columns of group h % 32
    val = torch.arange(I // 128, device="cuda") % 7 + 1
    up = (torch.eye(128, device="cuda", dtype=torch.int64)[None] * val[:, None, None]).view(I, H)
    grp = torch.arange(I, device="cuda") // 128
    down = (grp[None] == torch.arange(H, device="cuda")[:, None] % 32).long()
    t["w_up"].copy_(pack(torch, up).repeat(E))
    t["w_down"].copy_(pack(torch, down).repeat(E))
    t["s_up"].fill_(1.0)
    t["s_down"].fill_(1.0)
    tok = torch.arange(T, device="cuda")[:, None]
    idx = (tok * k + torch.arange(k, device="cuda")[None]) % E  # T k / E tokens per expert
    if crowded:  # every other token's first slot is expert 0: 64-token tiles
        idx[::2, 0] = 0
        idx[::2, 1:] = idx[::2, 1:].clamp(min=1)
    assert all(len(set(r)) == k for r in idx.tolist())
    idx = idx.int().contiguous()
    ws = ly.workspace(T)
    rows = torch.arange(T, device="cuda")
    for draw in range(6):
        x = torch.zeros(T, H, dtype=torch.bfloat16, device="cuda")
        x[rows, torch.randint(0, H, (T,), device="cuda", generator=g)] = (
            torch.randn(T, device="cuda", generator=g) * 4).to(torch.bfloat16)
        got = ly.experts(x, idx, ws)[:T * k]
        want = decode_rows(torch, ly, x, idx, ws)
        torch.cuda.synchronize()
        assert want.abs().max() > 1
        diff = int((got.view(torch.int16) != want.view(torch.int16)).sum())
        assert diff == 0, (draw, diff)
