"""HIP prefill attention (saga_prefill_attention) vs the oracle's restatement
of the reference prefill (attention/attention.py:13-53: SDPA over
repeat_kv-expanded key and value heads).

bf16 / f16 outputs against the float64 oracle on the same (rounded) inputs:
max-abs 2e-2 and rel-L2 5e-3.  P is rounded to the input dtype before the
P.V product, as in torch's flash kernels; transformers' own bf16 SDPA errors
are printed beside ours at the larger shapes.  Shapes cover asymmetric key /
value heads, lengths that are not multiples of the 64-key tile or the query
block, bool and float masks (broadcast over heads, wider than the keys),
non-causal calls, a causal chunk after cached positions (causal_offset), one
query, one key, f16, strided query / output views, and the reference-API
module's dispatch to the kernel."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import saga_oracle as O
from saga_amd import ops

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 5e-3


def _inputs(seed, b, q_h, k_h, v_h, Lq, Lk, d, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.float32).to(dtype)
    return mk(b, q_h, Lq, d), mk(b, k_h, Lk, d), mk(b, v_h, Lk, d)


def _np(t):
    return t.detach().to(torch.float64).cpu().numpy()


def _check(out, ref, what):
    got = _np(out)
    err_abs, err_l2 = float(np.max(np.abs(got - ref))), rel_l2(got, ref)
    print(f"{what}: max-abs {err_abs:.2e} rel-L2 {err_l2:.2e}", flush=True)
    assert np.isfinite(got).all(), what
    assert err_abs < MAX_ABS and err_l2 < REL_L2, (what, err_abs, err_l2)


CASES = [
    # b, q_h, k_h, v_h, Lq, Lk, d, causal
    (1, 12, 1, 2, 300, 300, 128, True),    # Qwen2.5-1.5B SAGA heads
    (2, 15, 1, 5, 200, 200, 64, True),     # SmolLM2-360M SAGA heads
    (1, 4, 2, 4, 130, 257, 128, False),    # more value heads than key heads, ragged
    (3, 6, 3, 2, 65, 65, 64, True),        # more key heads than value heads
    (1, 2, 1, 1, 1, 97, 128, False),       # one query
    (1, 2, 1, 2, 33, 1, 64, False),        # one key
    (2, 8, 8, 8, 129, 129, 128, True),     # plain multi-head
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "b{}_q{}k{}v{}_Lq{}_Lk{}_d{}_{}".format(
    *c[:7], "causal" if c[7] else "full"))
def test_prefill_matches_oracle(case):
    b, q_h, k_h, v_h, Lq, Lk, d, causal = case
    print(f"prefill {case}", flush=True)
    q, k, v = _inputs(1, b, q_h, k_h, v_h, Lq, Lk, d)
    out = ops.prefill_attention(q, k, v, is_causal=causal)
    torch.cuda.synchronize()
    assert out.shape == (b, Lq, q_h, d) and out.dtype == q.dtype
    _check(out, O.prefill(_np(q), _np(k), _np(v), None, None, causal), f"prefill {case}")


@pytest.mark.parametrize("mdt", [torch.bool, torch.float32, torch.bfloat16])
def test_prefill_masks(mdt):
    """Masks [b, 1, Lq, Lk + 5] (broadcast over heads, cut to the keys) and
    [1, q_h, Lq, Lk]: bool keeps True, float is added (SDPA semantics)."""
    b, q_h, k_h, v_h, Lq, Lk, d = 2, 6, 1, 3, 77, 140, 128
    print(f"prefill mask {mdt}", flush=True)
    q, k, v = _inputs(2, b, q_h, k_h, v_h, Lq, Lk, d)
    g = torch.Generator(device="cuda").manual_seed(3)
    for shape in ((b, 1, Lq, Lk + 5), (1, q_h, Lq, Lk)):
        r = torch.rand(*shape, generator=g, device="cuda")
        if mdt == torch.bool:
            m = r < 0.6
            m[..., 0] = True
        else:
            m = torch.where(r < 0.3, torch.full_like(r, -float("inf")), torch.randn_like(r)).to(mdt)
            m[..., 0] = 0
        m[..., 3, :] = False if mdt == torch.bool else -float("inf")  # a query that sees no key: 0
        out = ops.prefill_attention(q, k, v, attention_mask=m, scaling=0.1)
        torch.cuda.synchronize()
        ref = O.prefill(_np(q), _np(k), _np(v), m.cpu().numpy() if mdt == torch.bool else _np(m), 0.1, False)
        _check(out, ref, f"mask {mdt} {shape}")
        assert not out[:, 3].any()


def test_prefill_causal_offset_chunk():
    """A chunk of 50 queries after 250 cached positions: causal_offset 250
    equals the oracle with the explicit mask key <= 250 + i."""
    b, q_h, k_h, v_h, Lq, Lk, d = 1, 12, 1, 2, 50, 300, 128
    q, k, v = _inputs(4, b, q_h, k_h, v_h, Lq, Lk, d)
    out = ops.prefill_attention(q, k, v, is_causal=True, causal_offset=Lk - Lq)
    torch.cuda.synchronize()
    mask = np.arange(Lk)[None, None, None, :] <= (Lk - Lq + np.arange(Lq))[None, None, :, None]
    _check(out, O.prefill(_np(q), _np(k), _np(v), mask, None, False), "causal_offset 250")


def test_prefill_f16():
    q, k, v = _inputs(5, 2, 12, 1, 2, 190, 190, 128, dtype=torch.float16)
    out = ops.prefill_attention(q, k, v, is_causal=True)
    torch.cuda.synchronize()
    assert out.dtype == torch.float16
    _check(out, O.prefill(_np(q), _np(k), _np(v), None, None, True), "f16")


def test_prefill_strided_views():
    """The decoder's layout: queries [T, q_h, d] viewed as [1, q_h, T, d],
    caches [B, h, Lmax, d] cut to T, output written into a wider buffer."""
    T, q_h, d, Lmax = 333, 12, 128, 512
    g = torch.Generator(device="cuda").manual_seed(6)
    qt = torch.randn(T, q_h, d, generator=g, device="cuda").to(torch.bfloat16)
    kc = torch.randn(2, 1, Lmax, d, generator=g, device="cuda").to(torch.bfloat16)
    vc = torch.randn(2, 2, Lmax, d, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = qt.transpose(0, 1).unsqueeze(0), kc[1:2, :, :T], vc[1:2, :, :T]
    big = torch.full((1, T, q_h + 4, d), 7.0, device="cuda", dtype=torch.bfloat16)
    out = ops.prefill_attention(q, k, v, is_causal=True, out=big[:, :, 2:2 + q_h])
    torch.cuda.synchronize()
    assert out.data_ptr() == big[:, :, 2:].data_ptr()
    assert (big[:, :, :2] == 7).all() and (big[:, :, 2 + q_h:] == 7).all()
    _check(out, O.prefill(_np(q), _np(k), _np(v), None, None, True), "strided")


@pytest.mark.parametrize("L,d,q_h,k_h,v_h", [(4096, 128, 12, 1, 2), (2048, 64, 15, 1, 5)])
def test_prefill_long_vs_torch_fp32(L, d, q_h, k_h, v_h):
    """Long causal prefill vs torch SDPA in fp32 on the expanded heads (the
    oracle's float64 loop would take minutes at this size)."""
    print(f"prefill long L={L} d={d}", flush=True)
    q, k, v = _inputs(7, 1, q_h, k_h, v_h, L, L, d)
    out = ops.prefill_attention(q, k, v, is_causal=True)
    kx = k.float().repeat_interleave(q_h // k_h, dim=1)
    vx = v.float().repeat_interleave(q_h // v_h, dim=1)
    ref = torch.nn.functional.scaled_dot_product_attention(q.float(), kx, vx, is_causal=True).transpose(1, 2)
    tb = torch.nn.functional.scaled_dot_product_attention(q, kx.to(q.dtype), vx.to(q.dtype),
                                                          is_causal=True).transpose(1, 2)
    torch.cuda.synchronize()
    r = _np(ref)
    print(f"  torch bf16 SDPA: max-abs {float(np.max(np.abs(_np(tb) - r))):.2e} rel-L2 {rel_l2(_np(tb), r):.2e}")
    _check(out, r, f"long L={L} d={d}")


def test_reference_api_dispatches_to_the_kernel(monkeypatch):
    """sdpa_attention_forward (attention/attention.py:13-53) with a
    transformers-style module runs the HIP kernel for bf16 d-128 prefill and
    gives the expanded-SDPA result; fp32 operands keep torch SDPA."""
    from saga_amd.attention import attention as A
    calls = []
    real = ops.prefill_attention
    monkeypatch.setattr(ops, "prefill_attention", lambda *a, **kw: calls.append(1) or real(*a, **kw))

    class Mod(torch.nn.Module):
        num_key_value_groups = 6

    q, k, v = _inputs(8, 1, 12, 1, 2, 200, 200, 128)
    out, _ = A.sdpa_attention_forward(Mod(), q, k, v, None)
    torch.cuda.synchronize()
    assert calls and out.shape == (1, 200, 12, 128) and out.is_contiguous()
    _check(out, O.prefill(_np(q), _np(k), _np(v)), "reference API")
    calls.clear()
    out32, _ = A.sdpa_attention_forward(Mod(), q.float(), k.float(), v.float(), None)
    assert not calls
    assert rel_l2(_np(out32), _np(out)) < REL_L2


def test_prefill_rejects_bad_operands():
    q, k, v = _inputs(9, 1, 6, 4, 2, 16, 16, 128)  # 6 query heads over 4 key heads
    with pytest.raises(Exception, match="multiple"):
        ops.prefill_attention(q, k, v)
    q, k, v = _inputs(9, 1, 4, 1, 2, 16, 16, 128)
    m = torch.ones(1, 1, 16, 16, dtype=torch.bool, device="cuda")
    with pytest.raises(ValueError):
        ops.prefill_attention(q, k, v, attention_mask=m, is_causal=True)
    q96, k96, v96 = _inputs(9, 1, 4, 1, 2, 16, 16, 96)
    with pytest.raises(Exception, match="head_dim"):
        ops.prefill_attention(q96, k96, v96)


def _ref64(q, k, v, rows, causal, off, mask=None):
    """float64 attention of the given query rows: [b, len(rows), q_h, d]."""
    n = q.shape[1]
    k, v = (x.repeat_interleave(n // x.shape[1], 1).double() for x in (k, v))
    x = torch.matmul(q[:, :, rows].double(), k.transpose(2, 3)) / q.shape[3] ** 0.5
    if causal:
        keep = torch.arange(k.shape[2], device=q.device)[None, :] <= rows[:, None] + off
        x = x.masked_fill(~keep, float("-inf"))
    if mask is not None:
        m = mask[:, :, rows]
        x = x.masked_fill(~m, float("-inf")) if m.dtype == torch.bool else x + m.double()
    return torch.matmul(torch.softmax(x, -1).nan_to_num(0.0), v).transpose(1, 2)


# one launch per rule of the block shape: keys split (short grids, and chains of 1536 keys), 4 waves (short chains,
# d 64, below 8192 keys), 8 waves; lengths around the 64-key tile and the 128-key stage, queries and keys of unequal number
@pytest.mark.parametrize("b,q_h,k_h,v_h,d,Lq,Lk,causal,off", [
    (1, 2, 1, 1, 128, 1, 1, False, 0), (1, 3, 1, 3, 128, 129, 63, False, 0), (1, 4, 2, 1, 64, 65, 65, True, 0),
    (1, 12, 1, 2, 128, 127, 129, True, 2), (1, 12, 1, 2, 128, 1537, 1537, True, 0), (2, 15, 1, 5, 64, 1600, 1600, True, 0),
    (1, 12, 1, 2, 128, 70, 3011, False, 0), (1, 4, 1, 1, 64, 300, 1000, True, 700), (1, 4, 1, 1, 128, 300, 200, True, -150),
    (8, 12, 1, 2, 128, 321, 321, True, 0), (8, 15, 1, 5, 64, 200, 257, False, 0), (3, 24, 2, 2, 128, 1100, 1100, True, 0),
    # up to 320 (d 64) and 384 visible keys unsplit, then split; split stages that end inside either wave group's tile
    (1, 4, 2, 1, 64, 320, 320, True, 0), (1, 4, 2, 1, 64, 321, 321, True, 0), (1, 4, 2, 1, 128, 385, 385, True, 0), (1, 4, 1, 2, 128, 33, 449, False, 0),
    (1, 4, 1, 1, 128, 129, 511, False, 0), (1, 4, 1, 1, 64, 70, 513, False, 0), (1, 4, 1, 2, 128, 128, 900, True, 256),
    (1, 4, 1, 2, 128, 128, 900, True, 257), (1, 12, 1, 2, 128, 8200, 8200, True, 0), (1, 16, 1, 1, 128, 4200, 8255, False, 0), (1, 15, 1, 5, 64, 8193, 8193, True, 0)])
def test_prefill_block_shapes(b, q_h, k_h, v_h, d, Lq, Lk, causal, off):
    g = torch.Generator(device="cuda").manual_seed(Lq + Lk)
    q = torch.randn(b, Lq, q_h, d, generator=g, device="cuda").bfloat16().transpose(1, 2)
    # caches longer than Lk whose other rows are NaN: nothing past Lk may count
    cache = [torch.full((b, h, Lk + 130, d), float("nan"), device="cuda", dtype=torch.bfloat16) for h in (k_h, v_h)]
    for c in cache:
        c[:, :, :Lk] = torch.randn(c[:, :, :Lk].shape, generator=g, device="cuda").bfloat16()
    k, v = (c[:, :, :Lk] for c in cache)
    got = ops.prefill_attention(q, k, v, is_causal=causal, causal_offset=off)
    rows = torch.cat([torch.arange(min(Lq, 96)), torch.arange(max(Lq - 200, min(Lq, 96)), Lq)]).cuda()
    ref = _ref64(q, k, v, rows, causal, off)
    out = got[:, rows].double()
    # bf16 P and output: rel-L2 2e-3 as in the cases above, twice that as the bar
    assert torch.isfinite(out).all() and ((out - ref).norm() / ref.norm().clamp(min=1e-9)).item() < 5e-3


@pytest.mark.parametrize("kind", ["bool", "bytes", "half", "float", "strided", "strided half", "strided float"])
@pytest.mark.parametrize("b,h,d,Lq,Lk", [(2, 4, 64, 130, 191), (1, 2, 128, 257, 257), (3, 3, 128, 33, 64), (2, 2, 64, 5, 7)])
def test_prefill_mask_loads(kind, b, h, d, Lq, Lk):
    """Each way a mask reaches the kernel, rows at odd addresses, tiles wholly hidden, wholly visible and mixed,
    and queries that see nothing (0)."""
    g = torch.Generator(device="cuda").manual_seed(Lk)
    q, k, v = (torch.randn(b, h, L, d, generator=g, device="cuda").bfloat16() for L in (Lq, Lk, Lk))
    keep = torch.rand(b, 1, Lq, Lk + 3, generator=g, device="cuda") < 0.5
    keep[:, :, :, 64:128] = False
    keep[:, :, : Lq // 2, :64] = True
    keep[:, :, Lq // 3] = False
    keep = keep[..., :Lk]
    mask = keep
    if kind == "bytes":  # any non-zero byte keeps, as a cast to bool does
        mask = (keep.to(torch.uint8) * 5).view(torch.bool)
    elif kind.endswith(("half", "float")):
        mask = torch.randn(keep.shape, generator=g, device="cuda").masked_fill(~keep, float("-inf"))
        mask = mask.to(torch.bfloat16 if kind.endswith("half") else torch.float32)
    if kind.startswith("strided"):
        mask = mask.transpose(2, 3).contiguous().transpose(2, 3)
    got = ops.prefill_attention(q, k, v, mask).double()
    ref = _ref64(q, k, v, torch.arange(Lq, device="cuda"), False, 0, keep if mask.dtype == torch.bool else mask)
    assert ((got - ref).norm() / ref.norm()).item() < 5e-3 and not got[:, Lq // 3].any()


def test_prefill_far_rows():
    """Key rows 8 MB and more apart: a stage's offsets no longer fit the 32-bit lane offsets."""
    L, d = 90, 128
    buf = torch.zeros(L, 1 << 22, device="cuda", dtype=torch.bfloat16)
    k = buf[None, None, :, 64:64 + d]
    k.normal_()
    q, v = (torch.randn(1, n, L, d, device="cuda").bfloat16() for n in (2, 1))
    got = ops.prefill_attention(q, k, v, is_causal=True).double()
    ref = _ref64(q, k, v, torch.arange(L, device="cuda"), True, 0)
    assert ((got - ref).norm() / ref.norm()).item() < 5e-3


# the split-key, 4-wave and 8-wave blocks; lengths one past a 64-key tile (a stage filled up with repeated rows) and,
# for comparison, whole tiles
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["full", "causal", "bool", "half", "float"])
@pytest.mark.parametrize("b,q_h,Lq,Lk,d", [(1, 4, 70, 65, 64), (1, 4, 70, 65, 128), (2, 4, 33, 129, 64), (1, 4, 130, 129, 128),
                                           (1, 4, 70, 128, 128), (1, 4, 70, 385, 128), (2, 4, 33, 449, 64),
                                           (1, 4, 130, 513, 128), (1, 4, 70, 512, 128), (11, 12, 130, 129, 64), (11, 12, 130, 65, 128),
                                           (22, 12, 1, 8193, 128)])
def test_prefill_infinite_last_value(b, q_h, Lq, Lk, d, kind, dt):
    """An infinite value in the last key row makes that dim infinite for the queries that see the row: what a partial
    tile is filled up with has weight 0 and must not meet it."""
    g = torch.Generator(device="cuda").manual_seed(Lk + d)
    q, k, v = (torch.randn(b, h, L, d, generator=g, device="cuda").to(dt) for h, L in ((q_h, Lq), (1, Lk), (2, Lk)))
    v[:, 0, -1, 5], v[:, 1, -1, 6] = float("inf"), -float("inf")
    mask = None
    if kind in ("bool", "half", "float"):
        mask = torch.rand(b, 1, Lq, Lk, generator=g, device="cuda") < 0.7
        mask[..., -1] = True
        if kind != "bool":
            mask = torch.zeros(mask.shape, device="cuda").masked_fill(~mask, -float("inf"))
            mask = mask.to(dt) if kind == "half" else mask
    causal = kind == "causal"  # its last query sees the last key, the others do not
    got = ops.prefill_attention(q, k, v, mask, is_causal=causal, causal_offset=Lk - Lq if causal else 0)
    rows = torch.arange(Lq - 1 if causal else 0, Lq, device="cuda")
    ref = _ref64(q, k, v, rows, causal, Lk - Lq if causal else 0, mask)
    out, half = got[:, rows].double(), q_h // 2
    assert (out[:, :, :half, 5] == float("inf")).all() and (out[:, :, half:, 6] == -float("inf")).all()
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(out), fin)
    # 16-bit P and output, as in the cases above
    assert ((out[fin] - ref[fin]).norm() / ref[fin].norm()).item() < 5e-3
