"""The prompt's own kernels (16-byte vector forms of rmsnorm, silu_mul and
rope_kv_append; weight unpacking) at the edges of their vectors, tiles and
blocks, against float64 or the element-by-element form that unaligned rows
take."""
import pytest
import torch

from gpu_util import unpack_rows
from saga_amd import ops

pytestmark = pytest.mark.gpu
DTS = [torch.bfloat16, torch.float16]
HALF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}  # largest relative rounding error: half a unit of 8 / 11 bits


def _unaligned(t):
    """The same values in rows that start 2 bytes past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    out = buf[1:1 + t.numel()].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("N,H", [(1, 8), (3, 24), (4, 512), (5, 520), (2, 2056), (9, 1536), (3, 8192), (2, 8200), (3, 1004)])
def test_rmsnorm_rows(dt, N, H):
    g = torch.Generator(device="cuda").manual_seed(N * H)
    x = torch.randn(N, H, generator=g, device="cuda").to(dt)
    w = torch.randn(H, generator=g, device="cuda").to(dt)
    xd = x.double()
    want = w.double() * xd / torch.sqrt((xd * xd).mean(-1, keepdim=True) + 1e-6)
    for a in (x, _unaligned(x)):
        y = ops.rmsnorm(a, w, 1e-6)
        # one rounding to the storage type (half an ulp) and fp32 sums of H terms
        assert ((y.double() - want).abs() <= want.abs() * (HALF[dt] + 1e-5) + 1e-7).all()
    y = x.clone()
    ops.rmsnorm(y, w, 1e-6, out=y)  # in place
    assert torch.equal(y, ops.rmsnorm(x, w, 1e-6))


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("N,H", [(1, 8), (3, 24), (7, 2560), (2, 8960), (65, 1016), (3, 1004), (75000, 8), (25003, 24),
                                 (235, 2560), (67, 8960), (591, 1016), (599, 1004), (1, 600008)])
def test_silu_mul_rows(dt, N, H):
    g = torch.Generator(device="cuda").manual_seed(N + H)
    x = (torch.randn(N, 2 * H, generator=g, device="cuda") * 3).to(dt)
    xd = x.double()
    want = torch.nn.functional.silu(xd[:, :H]) * xd[:, H:]
    for a in (x, _unaligned(x)):
        y = ops.silu_mul(a)
        assert ((y.double() - want).abs() <= want.abs() * (HALF[dt] + 1e-5) + 1e-7).all()
    if dt == torch.bfloat16:  # the same arithmetic; f16's last product may round once (v_fma_mix) or twice
        assert torch.equal(y, ops.silu_mul(x))


def test_silu_mul_extremes():
    """exp(-gate) overflowing or vanishing, infinities and NaN as the element form gives them."""
    big = float(torch.finfo(torch.bfloat16).max)
    vals = [0.0, -0.0, 90.0, -90.0, big, -big, float("inf"), -float("inf"), float("nan"), 1.0]
    g = torch.tensor([v for v in vals for _ in vals] + [0.0] * 4, device="cuda").bfloat16()
    u = torch.tensor(vals * len(vals) + [0.0] * 4, device="cuda").bfloat16()
    x = torch.cat([g, u]).reshape(1, -1).repeat(6000, 1)  # the vector form's sizes
    torch.testing.assert_close(ops.silu_mul(x), ops.silu_mul(_unaligned(x)), rtol=0, atol=0, equal_nan=True)
    torch.testing.assert_close(ops.silu_mul(x)[:1], ops.silu_mul(x[:1]), rtol=0, atol=0, equal_nan=True)


def test_silu_mul_past_the_threads_of_a_launch():
    """2^35 and more outputs, all of one value, in rows 8 elements apart: only the last thread writes the last ones."""
    N, H = 65535, (1 << 19) + 2048
    x = torch.full((1, 2 * H), 1.5, device="cuda", dtype=torch.bfloat16)
    y = torch.zeros(8 * (N - 1) + H, device="cuda", dtype=torch.bfloat16)
    ops.silu_mul(x.expand(N, -1), out=y.as_strided((N, H), (8, 1)))
    assert bool((y == ops.silu_mul(x)[0, 0]).all())


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("N,n_q,n_k,n_v,d", [(1, 12, 1, 2, 128), (4, 15, 1, 5, 64), (5, 3, 1, 1, 16), (67, 12, 2, 2, 128),
                                             (6, 4, 2, 4, 48), (5, 2, 1, 1, 24),
                                             # 3072 (token, head) pairs and more: vectors, 1 token per block, 2 from 1536
                                             (205, 12, 1, 2, 128), (147, 15, 1, 5, 64), (613, 3, 1, 1, 16), (310, 4, 2, 4, 48),
                                             (1535, 3, 1, 1, 16), (1537, 12, 1, 2, 128), (1601, 2, 1, 1, 24)])
def test_rope_kv_append_rows(dt, N, n_q, n_k, n_v, d):
    g = torch.Generator(device="cuda").manual_seed(N + d)
    B, Lmax = 3, max(80, N)
    qkv = torch.randn(N, (n_q + n_k + n_v) * d, generator=g, device="cuda").to(dt)
    pos = torch.randperm(Lmax, generator=g, device="cuda")[:N].int()
    pos[N // 2] = Lmax if N > 4 else pos[N // 2]  # out of range: NaN queries, no cache row
    batch = (torch.arange(N, device="cuda") % B).int()
    got = []
    for rows in (qkv, _unaligned(qkv)):
        k = torch.zeros(B, n_k, Lmax, d, device="cuda", dtype=dt)
        v = torch.zeros(B, n_v, Lmax, d, device="cuda", dtype=dt)
        got.append((ops.rope_kv_append(rows, n_q, n_k, n_v, 1e4, pos, k, v, batch=batch), k, v))
    for a, b in zip(*got):
        torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True)
    assert bool(torch.isnan(got[0][0]).any()) == (N > 4)
    assert int((got[0][2] != 0).any(-1).sum()) == (N - (N > 4)) * n_v


@pytest.mark.parametrize("rows", [16, 8])
@pytest.mark.parametrize("N,K", [(16, 64), (48, 192), (32, 512), (64, 576), (1920, 1536), (32, 8960)])
def test_unpack_gemv_weights(rows, N, K):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    p = ops.pack_gemv_weight(w, rows)
    plain, pairs = ops.unpack_gemv_weights([p, p], [None, (1, N)])
    assert torch.equal(plain, w) and torch.equal(plain, unpack_rows(p))
    assert torch.equal(pairs, torch.cat([w[0::2], w[1::2]]))


def test_unpack_rotary_heads_and_errors():
    n_q, n_k, n_v, d, K = 3, 1, 2, 64, 128
    w = torch.randn((n_q + n_k + n_v) * d, K, device="cuda").bfloat16()
    p = ops.pack_gemv_weight(w[ops.rope_pair_order(n_q, n_k, n_v, d, device="cuda")].contiguous(), 8)
    a, b, c = ops.unpack_gemv_weights([p, w, p], [(n_q + n_k, d), None, None])
    assert torch.equal(a, w) and b is w and torch.equal(c, unpack_rows(p))
    for heads in ((7, d), (1, d - 1), (1, 80), (-1, d)):
        with pytest.raises(RuntimeError, match="unpack"):
            ops.unpack_gemv_weights([p], [heads])
    with pytest.raises(RuntimeError, match="unpack"):
        ops.unpack_gemv_weights([p] * 9)
