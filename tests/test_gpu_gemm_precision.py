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


@pytest.mark.parametrize("T", [40, 255, 256, 512, 1024])
def test_dots_are_as_near_as_the_decode_items(torch, T):
    """Gate dots that are 0 in 64 bits (every group's second half repeats x and
    negates the weights), read back as act = silu(e) * 1 = e / 2 of their fp32
    error e: at 17 tokens and more, in tiles of every height, the mean square is
    no larger than that of the decode items on the same tokens."""
    from ainfer_amd.moe import MoeLayer
    from ainfer_amd.synthetic import MoeConfig
    print(f"[case] dot error T={T}", flush=True)
    H, E, k, I = 2048, 64, 8, 256
    ly = MoeLayer(MoeConfig("dot", H, E, k, I, 0, (T,), seed=3))
    g = torch.Generator(device="cuda").manual_seed(1)
    t = ly.t
    q = torch.randint(-7, 8, (E * I, H // 128, 64), device="cuda", generator=g)
    t["w_gate"].copy_(pack(torch, torch.cat([q, -q], -1).view(E * I, H)))
    up = torch.zeros(I, H, dtype=torch.int64, device="cuda")
    up[:, 127] = 1
    down = (torch.arange(I, device="cuda")[None] == torch.arange(H, device="cuda")[:, None] % I).long()
    t["w_up"].copy_(pack(torch, up).repeat(E))
    t["w_down"].copy_(pack(torch, down).repeat(E))
    for n in ("s_gate", "s_up", "s_down"):
        t[n].fill_(1.0)
    x = torch.randn(T, H // 128, 64, device="cuda", generator=g)
    x[:, 0, 63] = 1  # column 127: what up reads
    x = torch.cat([x, x], -1).view(T, H).to(torch.bfloat16)
    idx = torch.stack([torch.randperm(E, device="cuda", generator=g)[:k] for _ in range(T)]).int()
    ws = ly.workspace(T)
    rms = [float(o.double().pow(2).mean().sqrt())
           for o in (ly.experts(x, idx, ws)[:T * k], decode_rows(torch, ly, x, idx, ws))]
    print(f"[dot error] T={T} gemm {rms[0]:.2e} items {rms[1]:.2e}", flush=True)
    assert 0 < rms[0] <= rms[1], rms
