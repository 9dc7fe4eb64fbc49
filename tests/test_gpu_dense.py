"""Dense split-L decode on the GPU vs the oracle (full_einsum_forward,
attention/attention.py:64-85), including the dense-GQA comparator shape."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from gpu_util import host, qkv, randn
from oracle import saga_oracle as O
from saga_amd import ops

pytestmark = pytest.mark.gpu

SHAPES = [  # b, q_h, k_h, v_h, d, L
    (1, 15, 1, 5, 64, 4096),
    (2, 12, 1, 2, 128, 1000),
    (2, 12, 2, 2, 128, 777),
    (3, 6, 2, 3, 128, 257),
    (1, 8, 8, 8, 64, 40),
    (2, 12, 2, 1, 128, 300),
    (8, 12, 2, 2, 128, 33024),
    # one key head below batch 4: the query heads split over two units that
    # read the same key head (each half spanning two value heads; one each)
    (1, 12, 1, 4, 64, 5000),
    (3, 16, 1, 2, 128, 2500),
]


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_dense_matches_oracle(dt, shape):
    b, q_h, k_h, v_h, d, L = shape
    print(f"dense dt={dt} shape={shape}", flush=True)
    rng = np.random.default_rng(sum(shape) + 1)
    (q, k, v), (qd, kd, vd) = qkv(rng, b, q_h, k_h, v_h, d, L, dt, qscale=2.0)
    out32 = host(ops.dense_decode(qd, kd, vd, out_dtype=torch.float32))
    ref = O.dense(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64))
    assert rel_l2(out32, ref) < (1e-5 if dt == "f32" else 1e-4)
    if dt != "f32":
        out16 = host(ops.dense_decode(qd, kd, vd))
        assert np.max(np.abs(out16 - ref)) < 2e-2


def test_dense_with_masks():
    rng = np.random.default_rng(5)
    b, q_h, k_h, v_h, d, L = 2, 12, 1, 2, 128, 600
    (q, k, v), (qd, kd, vd) = qkv(rng, b, q_h, k_h, v_h, d, L, "bf16")
    valid = rng.random((b, 1, 1, L + 3)) > 0.3
    for m in (valid, np.where(valid, 0.0, -np.inf).astype(np.float32)):
        out = host(ops.dense_decode(qd, kd, vd, torch.from_numpy(m).cuda(), 0.1, out_dtype=torch.float32))
        ref = O.dense(q, k, v, m, 0.1)
        assert rel_l2(out, ref) < 1e-4


def test_workspace_reuse_across_shapes():
    """Calls of different shapes share one cached workspace; the arrival
    counters live in a fixed region, so a later call never sees stale data
    of an earlier layout (regression test)."""
    rng = np.random.default_rng(6)
    shapes = [(8, 12, 2, 2, 128, 20000), (2, 12, 1, 2, 128, 1000), (1, 15, 1, 5, 64, 4096), (2, 12, 1, 2, 128, 1000)]
    for shape in shapes:
        b, q_h, k_h, v_h, d, L = shape
        (q, k, v), (qd, kd, vd) = qkv(rng, b, q_h, k_h, v_h, d, L, "bf16")
        out = host(ops.dense_decode(qd, kd, vd, out_dtype=torch.float32))
        assert rel_l2(out, O.dense(q, k, v)) < 1e-4, shape
        table = torch.full((b * q_h,), 2e-4, device="cuda")
        fast = host(ops.atopn_decode(qd, kd, vd, table, 128, out_dtype=torch.float32))
        ref, _, _, _ = O.fast(q, k, v, host(table), None, 128, None)
        assert rel_l2(fast, ref) < 1e-3, shape


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("mask_kind", [None, "bool", "float"])
def test_full_einsum_forward_several_queries(dt, mask_kind):
    """full_einsum_forward with l_q > 1 (attention/attention.py:64-85): every
    query attends to all keys plus the mask (is_causal is ignored, as in the
    reference), query head h reading key head h // (q_h / k_h) and value
    head h // (q_h / v_h); a bool mask adds 1.0 where true."""
    from saga_amd.attention import attention as A
    rng = np.random.default_rng(17 + (mask_kind is not None))
    b, q_h, k_h, v_h, d, L, l_q = 3, 12, 1, 2, 128, 700, 5
    q, qd = randn(rng, (b, q_h, l_q, d), dt)
    (_, k, v), (_, kd, vd) = qkv(rng, b, q_h, k_h, v_h, d, L, dt)
    m = None
    if mask_kind == "bool":
        m = rng.random((b, 1, l_q, L + 4)) > 0.4
    elif mask_kind == "float":
        m = rng.standard_normal((1, q_h, l_q, L), dtype=np.float32)
    md = None if m is None else torch.from_numpy(m).cuda()
    out = A.full_einsum_forward(qd, kd, vd, md, is_causal=True, scaling=0.09)
    assert tuple(out.shape) == (b, q_h, l_q, d) and out.dtype == qd.dtype
    ref = O.dense(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), m, 0.09)
    got = host(out)
    assert rel_l2(got, ref) < (1e-5 if dt == "f32" else 5e-3)
    if dt != "f32":
        assert np.max(np.abs(got - ref)) < 2e-2


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("b,q_h,k_h,v_h,d", [(4, 12, 2, 2, 128), (4, 12, 1, 2, 128), (4, 8, 2, 1, 128), (5, 15, 1, 5, 64),
                                             (4, 16, 4, 8, 64), (2, 16, 1, 1, 64), (4, 12, 1, 3, 128)])
@pytest.mark.parametrize("L", [1, 31, 33, 129, 1055])
def test_dense_value_head_layouts(dt, b, q_h, k_h, v_h, d, L):
    """Units of one, two and five whole value heads (MFMA) and others (VALU), at the edges of the 32-position step, with
    ragged kv_len: cache rows past it are NaN (VALU: large) and one value head holds infinities, which reach its own
    query heads only."""
    import torch as T
    g = T.Generator(device="cuda").manual_seed(L + q_h)
    tdt = T.bfloat16 if dt == "bf16" else T.float16
    q = T.randn(b, q_h, 1, d, generator=g, device="cuda").to(tdt)
    k = T.randn(b, k_h, L + 40, d, generator=g, device="cuda").to(tdt)
    v = T.randn(b, v_h, L + 40, d, generator=g, device="cuda").to(tdt)
    lens = [max(1, L - 7 * i) for i in range(b)]
    for i, n in enumerate(lens):
        k[i, :, n:] = v[i, :, n:] = float("nan") if v_h != 3 else 100.0
    if v_h != 3:
        v[:, 0, 0] = float("inf")
    kv = T.tensor(lens, dtype=T.int32, device="cuda")
    out = ops.dense_decode(q, k[:, :, :L], v[:, :, :L], kv_len=kv, out_dtype=T.float32).double()
    for i, n in enumerate(lens):
        kk = k[i, :, :n].double().repeat_interleave(q_h // k_h, 0)
        vv = v[i, :, :n].double().repeat_interleave(q_h // v_h, 0)
        p = T.softmax((q[i].double() @ kk.transpose(1, 2)) / d ** 0.5, -1)
        ref = (p @ vv)[:, 0]
        own = T.arange(q_h) < q_h // v_h  # the query heads of value head 0
        assert v_h == 3 or T.isinf(out[i, own, 0]).all()
        if v_h > 1:
            # exact products, fp32 sums and exp: 1e-6 relative and a few units per sum
            got, want = out[i, ~own, 0], ref[~own]
            assert T.isfinite(got).all() and ((got - want).norm() / want.norm()).item() < 1e-5


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("q_h,k_h,v_h,d", [(12, 2, 2, 128), (12, 1, 2, 128), (15, 1, 5, 64), (12, 1, 3, 128)])
@pytest.mark.parametrize("L,gap", [(33, 12.0), (4096, 17.0), (4096, 28.0), (20000, 40.0)])
def test_dense_dominating_keys(dt, q_h, k_h, v_h, d, L, gap):
    """Keys `gap` nats above the rest (in every wave's range) whose values are 0, as attention sinks have: the output is
    what the small weights give, in either type held to 24 bits."""
    import torch as T
    b = 8
    g = T.Generator(device="cuda").manual_seed(L + q_h)
    tdt = T.bfloat16 if dt == "bf16" else T.float16
    q, k, v = (T.randn(b, h, n, d, generator=g, device="cuda") for h, n in ((q_h, 1), (k_h, L), (v_h, L)))
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[:, :, ::32] = 0.0
    k[:, :, ::32, 0] = gap * d ** 0.5 / 8.0
    v += 0.5
    v[:, :, ::32] = 0.0
    q, k, v = q.to(tdt), k.to(tdt), v.to(tdt)
    out = ops.dense_decode(q, k, v, out_dtype=T.float32).double()
    for i in range(b):
        kk, vv = k[i].double().repeat_interleave(q_h // k_h, 0), v[i].double().repeat_interleave(q_h // v_h, 0)
        ref = (T.softmax((q[i].double() @ kk.transpose(1, 2)) / d ** 0.5, -1) @ vv)[:, 0]
        # logits of up to 40 rounded to fp32 and exp of them: 40 * 2^-23 = 5e-6 per weight
        assert ((out[i, :, 0] - ref).norm() / ref.norm()).item() < 1e-5


LAYOUTS = [(4, 12, 2, 2, 128), (4, 12, 1, 2, 128), (4, 8, 2, 1, 128), (5, 15, 1, 5, 64), (4, 16, 4, 8, 64), (2, 16, 1, 1, 64),
           (4, 12, 1, 3, 128), (4, 16, 1, 4, 64)]


def _dense64(q, k, v, x_add):
    """float64 attention of one batch row: q [q_h, 1, d], k / v [h, n, d], x_add [1 or q_h, n] added to the logits."""
    q_h, _, d = q.shape
    kk, vv = (t.double().repeat_interleave(q_h // t.shape[0], 0) for t in (k, v))
    x = (q.double() @ kk.transpose(1, 2))[:, 0] / d ** 0.5 + x_add
    return (torch.softmax(x, -1)[:, None] @ vv)[:, 0]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mask", [None, "bool", "float", "heads"])
@pytest.mark.parametrize("b,q_h,k_h,v_h,d", LAYOUTS)
@pytest.mark.parametrize("L", [1, 33, 1055])
def test_dense_value_head_layouts_numeric(dt, mask, b, q_h, k_h, v_h, d, L):
    """Every head of every layout against 64 bits, with ragged kv_len and with masks (bool adds 1, as the reference does;
    float broadcast or per head, with -inf)."""
    g = torch.Generator(device="cuda").manual_seed(L + q_h + d)
    q, k, v = (torch.randn(b, h, n, d, generator=g, device="cuda").to(dt) for h, n in ((q_h, 1), (k_h, L), (v_h, L)))
    lens = [max(1, L - 9 * i) for i in range(b)]
    m = None
    if mask == "bool":
        m = torch.rand(b, 1, 1, L, generator=g, device="cuda") < 0.5
    elif mask:
        m = torch.randn(b, q_h if mask == "heads" else 1, 1, L, generator=g, device="cuda")
        m[torch.rand(m.shape, generator=g, device="cuda") < 0.3] = float("-inf")
        m[..., 0] = 0.0
    kv = torch.tensor(lens, dtype=torch.int32, device="cuda")
    out = ops.dense_decode(q, k, v, m, kv_len=kv, out_dtype=torch.float32).double()
    for i, n in enumerate(lens):
        add = 0.0 if m is None else m[i, :, 0, :n].double()
        ref = _dense64(q[i], k[i, :, :n], v[i, :, :n], add)
        # fp32 scores, exp and sums: a few 2^-24 per term
        assert ((out[i, :, 0] - ref).norm() / ref.norm()).item() < 1e-5


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,q_h,k_h,v_h,d", [c for c in LAYOUTS if c[3] not in (3, 4)])
@pytest.mark.parametrize("L", [1, 40, 700])
def test_dense_special_values(dt, b, q_h, k_h, v_h, d, L):
    """inf, -inf, both, NaN, and an infinite value of weight 0 (NaN), each in a dim of its own of the last value head; all
    other dims and heads are compared."""
    g = torch.Generator(device="cuda").manual_seed(L + q_h)
    q, k, v = (torch.randn(b, h, n, d, generator=g, device="cuda").to(dt) for h, n in ((q_h, 1), (k_h, L), (v_h, L)))
    inf = float("inf")
    v[:, -1, 0, 3], v[:, -1, L // 2, 4], v[:, -1, L - 1, 7] = inf, -inf, float("nan")
    v[:, -1, 0, 5], v[:, -1, L - 1, 5] = inf, -inf  # one value where L is 1: -inf
    add = torch.zeros(b, 1, 1, L, device="cuda")
    if L > 1:
        add[..., 1] = -inf
        v[:, -1, 1, 9] = inf
    out = ops.dense_decode(q, k, v, add, out_dtype=torch.float32).double()
    for i in range(b):
        ref = _dense64(q[i], k[i], v[i], add[i, :, 0].double())
        torch.testing.assert_close(out[i, :, 0], ref, rtol=0, atol=1e-5, equal_nan=True)
        own = ref[q_h - q_h // v_h:]  # the special values' own query heads, and no others
        assert (own[:, 3] == inf).all() and (own[:, 4] == -inf).all() and own[:, 7].isnan().all()
        assert own[:, 5].isnan().all() if L > 1 else (own[:, 5] == -inf).all()
        assert torch.isfinite(ref[: q_h - q_h // v_h]).all() and (L == 1 or own[:, 9].isnan().all())
