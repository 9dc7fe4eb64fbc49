"""The prompt's fused gate/up projection + SiLU against float64 (GPU)."""
import pytest
import torch

from saga_amd import ops

pytestmark = pytest.mark.gpu

# token counts at the edges of a block (128 and 256 tokens), weights of one tile and of a partial last block (128 and
# 256 rows), one k step, odd and even numbers of them; the launch takes blocks of 128 x 128 but for (700, 17936) and
# (2500, 4112): 256 x 256, (2111, 2576): 256 x 128, and (1000, 17936), (2100, 7952): 256 x 256 with a
# rest in halves, the second with a last half past the weight's rows
CASES = [(1, 16, 64), (17, 144, 192), (64, 5120, 960), (65, 272, 128), (128, 640, 64), (129, 5136, 320), (512, 1008, 448),
         (513, 272, 1536), (768, 5136, 192), (700, 17936, 192), (2500, 4112, 64), (2111, 2576, 960),
         (1000, 17936, 128), (2100, 7952, 64)]


@pytest.mark.parametrize("T,N,K", CASES)
@pytest.mark.parametrize("strided", [False, True])
def test_prompt_mlp(T, N, K, strided):
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    x = torch.randn(T, K + (8 if strided else 0), generator=g, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(N, K, generator=g, device="cuda") * (2.0 / K ** 0.5)).bfloat16()
    out = torch.full((T, N // 2 + (8 if strided else 0)), 7.0, device="cuda", dtype=torch.bfloat16)
    got = ops.prompt_mlp(x, ops.pack_gemv_weight(w), out=out[:, : N // 2])
    xd, wd = x.double().cpu(), w.double().cpu()
    p, bound = xd @ wd.t(), (xd.abs() @ wd.t().abs()) * (K * 2.0 ** -24)  # fp32 sums of K products
    gate, up, eg, eu = p[:, 0::2], p[:, 1::2], bound[:, 0::2], bound[:, 1::2]
    silu = gate * torch.sigmoid(gate)
    want = silu * up
    # |silu'| <= 1.1; one bf16 rounding (half a unit of 8 bits, 2^-8 at most) and the fp32 activation's 8e-6
    tol = want.abs() * (2.0 ** -8 + 1e-5) + 1.1 * eg * (up.abs() + eu) + silu.abs() * eu + 1e-30
    assert bool(((got.double().cpu() - want).abs() <= tol).all())
    if strided:
        assert bool((out[:, N // 2:] == 7.0).all())


def test_prompt_mlp_special_values():
    """Gates far below and above: silu goes to 0 and to the gate; a NaN row stays its own."""
    K, N, T = 64, 32, 70
    x = torch.zeros(T, K, device="cuda", dtype=torch.bfloat16)
    x[0, 0], x[1, 0], x[2, 0] = -200.0, 200.0, float("nan")
    w = torch.zeros(N, K, device="cuda", dtype=torch.bfloat16)
    w[0::2, 0], w[1::2, 0] = 1.0, 0.5
    y = ops.prompt_mlp(x, ops.pack_gemv_weight(w)).float()
    assert bool((y[0] == 0).all()) and bool((y[1] == 20000).all() or ((y[1] - 20000).abs() <= 64).all())
    assert bool(y[2].isnan().all()) and bool((y[3:] == 0).all())


def test_prompt_mlp_vanishing_gates():
    """silu where 1 / (1 + exp(-gate)) is a subnormal number (gates of -87.4 to -88.7) and around."""
    K, N = 64, 32
    gates = torch.cat([torch.arange(-89.0, -80.0, 0.5), torch.arange(-80.0, 20.0, 1.0)]).cuda()
    x = torch.zeros(len(gates), K, device="cuda", dtype=torch.bfloat16)
    x[:, 0], x[:, 1] = gates, 1.0
    w = torch.zeros(N, K, device="cuda", dtype=torch.bfloat16)
    w[0::2, 0], w[1::2, 1] = 1.0, 2.0 ** 100
    y = ops.prompt_mlp(x, ops.pack_gemv_weight(w)).double()
    g = gates.bfloat16().double()
    want = (g * torch.sigmoid(g) * 2.0 ** 100)[:, None]
    # one rounding to bf16 (2^-8 at most) and the fp32 activation's 8e-6; below -88.7 exp overflows and silu is 0
    fine = (g > -88.7)[:, None]
    assert bool((((y - want).abs() <= want.abs() * (2.0 ** -8 + 1e-5)) | ~fine).all())


def test_prompt_mlp_refuses():
    x = torch.zeros(4, 96, device="cuda", dtype=torch.bfloat16)
    w = ops.pack_gemv_weight(torch.zeros(32, 96, device="cuda", dtype=torch.bfloat16))
    assert not ops.prompt_mlp_supported(w)
    with pytest.raises(Exception):
        ops.prompt_mlp(x, w)  # K % 64
    w = ops.pack_gemv_weight(torch.zeros(32, 64, device="cuda", dtype=torch.bfloat16))
    with pytest.raises(Exception):
        ops.prompt_mlp(x[:, :64].float(), w)
    with pytest.raises(Exception):
        ops.prompt_mlp(x[:, 1:65], w)  # rows not 16-byte aligned
