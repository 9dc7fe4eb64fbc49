"""The calls whose speed counts, on one MI355X: decode attention (Atop-N fast and calibration steps, dense), prefill
attention, the decode projections, a whole decode step and a whole prompt.

Decode-path cases replay a HIP graph captured in prepare(), as the decoder and a server do for every token; the
drop-in attention module ("call") and the prefill cases run eagerly, as transformers and a prompt do.

Head layouts and widths are those of the decoder shapes in saga_amd/decoder.py (Qwen2.5-1.5B and SmolLM2-360M, each
with SAGA's separate key / value heads and as plain GQA); lengths, batches and N are those of bench.py and of the
latency grid of saga_amd/speedup.py (batch 1-32, 4k-128k positions, N 128-2048).
"""
import math

import torch

import attention.attention as A
from saga_amd import ops
from saga_amd.decoder import (QWEN25_15B_GQA, QWEN25_15B_SAGA, SMOLLM2_360M_GQA, SMOLLM2_360M_SAGA, SagaDecoder,
                              gemv_tile_rows)

SHAPES = {"qwen": QWEN25_15B_SAGA, "qwen_gqa": QWEN25_15B_GQA, "smollm": SMOLLM2_360M_SAGA,
          "smollm_gqa": SMOLLM2_360M_GQA}
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
DEV = "cuda"

PROJ_LAYERS = 2      # decode layers per pass of a "proj" case: their weights exceed what the last-level cache keeps
PROJ_POSITIONS = 64  # cache length of a "proj" case: one row of it is written per token


def listed():
    return [
        # One layer of the smallest model at batch 1 through the reference's module API, launched eagerly as an
        # evaluation harness does (bench.py's C1 attention shape): host and launch latency.
        {"name": "call_b1_4k", "kind": "call", "shape": "smollm", "b": 1, "L": 4096, "N": 128, "dtype": "bf16", "mask": False},
        # The headline fast step of one layer: bench.py's default decode (static cache, 32769 filled positions).
        {"name": "atopn_b8_32k", "kind": "atopn", "shape": "qwen", "b": 8, "L": 33024, "fill": 32769, "N": 512,
         "dtype": "bf16", "peaked": False},
        # The reference's default latency grid: batch 32 at 64k, the largest decode attention call.
        {"name": "atopn_b32_64k", "kind": "atopn", "shape": "qwen", "b": 32, "L": 65544, "fill": 65541, "N": 512,
         "dtype": "bf16", "peaked": False},
        # The first decode step after a prompt: exact top-N and its threshold, at the headline shape ...
        {"name": "calibrate_b8_32k", "kind": "calibrate", "shape": "qwen", "b": 8, "L": 33024, "fill": 32769, "N": 512,
         "dtype": "bf16", "peaked": False},
        # ... and at 128k positions with N = 1024 (bench.py's long-context comparison), in f16.
        {"name": "calibrate_b4_128k", "kind": "calibrate", "shape": "qwen", "b": 4, "L": 131080, "fill": 131073,
         "N": 1024, "dtype": "f16", "peaked": False},
        # Dense decode of the plain GQA model at the headline shape: the comparator, and every "full" mode layer.
        {"name": "dense_gqa_b8_32k", "kind": "dense", "shape": "qwen_gqa", "b": 8, "L": 33024, "fill": 32769, "dtype": "bf16"},
        # Dense decode of the small model's many value heads over a ragged batch: exempt layers of a served batch.
        {"name": "dense_b4_8k_ragged", "kind": "dense", "shape": "smollm", "b": 4, "L": 8195, "fill": 0, "dtype": "bf16"},
        # Prompt attention of one layer, 32k causal (bench.py --prefill).
        {"name": "attn_b1_32k", "kind": "attn", "shape": "qwen", "b": 1, "T": 32768, "masked": False, "dtype": "bf16"},
        # Prompt attention of a left-padded evaluation batch: transformers passes a boolean causal + padding mask.
        {"name": "attn_b4_masked", "kind": "attn", "shape": "smollm", "b": 4, "T": 1021, "masked": True, "dtype": "bf16"},
        # Everything of a decode layer but its attention: o, gate/up + SiLU, down, q/k/v + RoPE + cache append.
        {"name": "proj_b8", "kind": "proj", "shape": "qwen", "b": 8},
        # A whole decode step of the headline model and cache: 28 layers, LM head and greedy token in one graph.
        {"name": "decode_b8_32k", "kind": "decode", "shape": "qwen", "b": 8, "L": 32768, "N": 512},
        # A whole prompt through the headline model: what a request waits for before its first token.
        {"name": "prompt_4k", "kind": "prompt", "shape": "qwen", "T": 4001},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "atopn", "atopn", "calibrate", "dense", "attn", "attn", "proj", "decode", "prompt"])
    if kind == "call":
        return {"kind": kind, "shape": rng.choice(["qwen", "smollm"]), "b": _log(rng, 1, 4), "L": _log(rng, 300, 8200),
                "N": rng.choice([64, 128, 256, 512]), "dtype": rng.choice(["bf16", "bf16", "f16"]),
                "mask": rng.random() < 0.3}
    if kind in ("atopn", "calibrate", "dense"):
        b = _log(rng, 1, 32)
        L = _log(rng, 2000, min(132000, 2000000 // b))
        c = {"kind": kind, "shape": rng.choice(["qwen", "qwen", "smollm", "qwen_gqa"]), "b": b, "L": L,
             "fill": rng.choice([0, L, L - L // 50]), "dtype": rng.choice(["bf16", "bf16", "bf16", "f16"])}
        if kind != "dense":
            c["N"] = rng.choice([128, 256, 512, 512, 1024, 2048])
            c["peaked"] = rng.random() < 0.2
        return c
    if kind == "attn":
        b = _log(rng, 1, 8)
        masked = rng.random() < 0.3
        return {"kind": kind, "shape": rng.choice(["qwen", "smollm", "qwen_gqa"]), "b": b,
                "T": _log(rng, 100, (3000 if masked else 30000) / math.sqrt(b)), "masked": masked,
                "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "proj":
        return {"kind": kind, "shape": rng.choice(["qwen", "qwen", "smollm"]), "b": _log(rng, 1, 32)}
    if kind == "decode":
        b = _log(rng, 1, 32)
        return {"kind": kind, "shape": rng.choice(["qwen", "smollm"]), "b": b, "L": _log(rng, 1000, 262144 // b),
                "N": rng.choice([128, 256, 512])}
    return {"kind": kind, "shape": rng.choice(["qwen", "smollm"]), "T": _log(rng, 128, 4000)}


# ------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *size, dtype=torch.float32, std=1.0):
    x = torch.randn(*size, generator=g, device=DEV, dtype=dtype)
    return x if std == 1.0 else x.mul_(std)


def _kv_lens(c):
    """Filled positions per batch row: all the same, or (fill 0) ragged from the whole cache down to a quarter."""
    b, L, fill = c["b"], c["L"], c.get("fill", c["L"])
    return [fill] * b if fill else [L - (3 * L // 4) * i // b for i in range(b)]


def _decode_inputs(c, seed):
    """q, k, v, filled lengths, additive mask and, for a fast step, the thresholds p* that the calibration of an
    earlier token's query left: N-th largest probability per (batch row, head)."""
    s, dt, b, L = SHAPES[c["shape"]], DTYPES[c["dtype"]], c["b"], c["L"]
    g = _gen(seed)
    q = _randn(g, b, s.n_q, 1, s.head_dim)
    # the next token's query is near the calibration token's, as measured in generations
    q_before = (0.9 * q + math.sqrt(1 - 0.81) * _randn(g, *q.shape)).to(dt)
    k = _randn(g, b, s.n_k, L, s.head_dim, dtype=dt)
    v = _randn(g, b, s.n_v, L, s.head_dim, dtype=dt)
    if c.get("peaked"):  # 1 % of the keys eight times as long: heads with a few dominating positions
        k.mul_(1 + 7 * (torch.rand(b, s.n_k, L, 1, generator=g, device=DEV) < 0.01).to(dt))
    q, lens = q.to(dt), _kv_lens(c)
    mask = None
    if c.get("mask"):  # left padding of an evaluation batch: row i hides its first i * L / 8 positions
        mask = torch.zeros(b, 1, 1, L, dtype=dt, device=DEV)
        for i in range(b):
            mask[i, ..., : i * L // 8] = torch.finfo(dt).min
    pstar = None
    if c["kind"] in ("atopn", "call"):
        rows = []
        for i in range(b):
            p = torch.softmax(_logits64(q_before, k, mask, i, lens[i]), dim=-1)
            rows.append(p.topk(min(c["N"], lens[i]), dim=-1).values[:, -1])
        pstar = torch.stack(rows).reshape(-1).float()
    return s, q, k, v, lens, mask, pstar


def _graphed(fn):
    """fn's launches as a HIP graph (after a warm-up on a side stream)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


def _bytes(n):
    return torch.empty(max(int(n), 256), dtype=torch.uint8, device=DEV)


def _prepare_decode_attention(c, seed):
    s, q, k, v, lens, mask, pstar = _decode_inputs(c, seed)
    if c["kind"] == "call":
        return {"q": q, "k": k, "v": v, "mask": mask, "table": pstar.reshape(1, -1).contiguous(), "N": c["N"]}
    b, L, d = c["b"], c["L"], s.head_dim
    kv_len = torch.tensor(lens, dtype=torch.int32, device=DEV)
    out = torch.empty_like(q)
    if c["kind"] == "dense":
        ws = _bytes(ops._lib.load().saga_dense_workspace_bytes(b, s.n_q, L, d))
        outs = {"out": out}

        def call():
            ops.dense_decode(q, k, v, kv_len=kv_len, out=out, workspace=ws)
    elif c["kind"] == "calibrate":
        ws = _bytes(ops.atopn_workspace_bytes(b, s.n_q, s.n_k, L, d, c["N"], True))
        thr = torch.empty(b * s.n_q, dtype=torch.float32, device=DEV)
        outs = {"out": out, "thr": thr}

        def call():
            ops.atopn_calibrate(q, k, v, c["N"], thr, kv_len=kv_len, out=out, workspace=ws)
    else:
        ws = _bytes(ops.atopn_workspace_bytes(b, s.n_q, s.n_k, L, d, c["N"]))
        outs = {"out": out}

        def call():
            ops.atopn_decode(q, k, v, pstar, c["N"], kv_len=kv_len, out=out, workspace=ws)
    return {"graph": _graphed(call), "outs": outs, "keep": (call, ws)}


def _attn_inputs(c, seed):
    s, dt, b, T = SHAPES[c["shape"]], DTYPES[c["dtype"]], c["b"], c["T"]
    g = _gen(seed)
    # [b, T, heads, d] projections viewed as [b, heads, T, d], as a model hands them over
    q, k, v = (_randn(g, b, T, h, s.head_dim, dtype=dt).transpose(1, 2) for h in (s.n_q, s.n_k, s.n_v))
    mask = None
    if c["masked"]:
        ar = torch.arange(T, device=DEV)
        pad = torch.tensor(_pads(c), device=DEV)
        mask = (ar[None, :] <= ar[:, None])[None, None] & (ar[None, None, None, :] >= pad[:, None, None, None])
    return s, q, k, v, mask


def _pads(c):
    """Left padding per row of a masked batch: none up to a half."""
    return [c["T"] * i // (2 * c["b"]) for i in range(c["b"])]


class _Attention(torch.nn.Module):
    num_key_value_groups = 1


def _weights(s, seed):
    """Random weights of a decoder in the layout SagaDecoder(weights=...) takes."""
    g, dt = _gen(seed), torch.bfloat16
    n = range(s.layers)

    def w(*size):
        return _randn(g, *size, dtype=dt, std=0.02)

    # unit-variance embeddings: as in a trained model, a layer's update is small beside the residual stream it joins
    # (a stream of 0.02 would be mostly the first layer's attention output, whose top-N cut turns bf16 rounding of
    # the query into percents)
    return {"embed": _randn(g, s.vocab, s.hidden, dtype=dt), "lm_head": None, "ln_f": (1 + w(s.hidden)),
            "ln1": [1 + w(s.hidden) for _ in n], "ln2": [1 + w(s.hidden) for _ in n],
            "w_qkv": [w(s.qkv_width, s.hidden) for _ in n],
            "b_qkv": [w(s.qkv_width) if s.qkv_bias else torch.zeros(s.qkv_width, device=DEV, dtype=dt) for _ in n],
            "w_o": [w(s.hidden, s.n_q * s.head_dim) for _ in n], "w_gu": [w(2 * s.intermediate, s.hidden) for _ in n],
            "w_d": [w(s.hidden, s.intermediate) for _ in n]}


def _proj_inputs(c, seed):
    s, b, dt = SHAPES[c["shape"]], c["b"], torch.bfloat16
    g = _gen(seed)
    layers = []
    for _ in range(PROJ_LAYERS):
        layers.append({"w_o": _randn(g, s.hidden, s.n_q * s.head_dim, dtype=dt, std=0.02),
                       "w_gu": _randn(g, 2 * s.intermediate, s.hidden, dtype=dt, std=0.02),  # rows gate_0, up_0, ...
                       "w_d": _randn(g, s.hidden, s.intermediate, dtype=dt, std=0.02),
                       "w_qkv": _randn(g, s.qkv_width, s.hidden, dtype=dt, std=0.02),
                       "b_qkv": _randn(g, s.qkv_width, dtype=dt, std=0.02),
                       "attn": _randn(g, b, s.n_q * s.head_dim, dtype=dt, std=0.1)})
    pos = torch.arange(b, device=DEV, dtype=torch.int32) % PROJ_POSITIONS
    return s, _randn(g, b, s.hidden, dtype=dt), layers, pos


def _prepare_proj(c, seed):
    s, x0, layers, pos = _proj_inputs(c, seed)
    b, d, dt = c["b"], s.head_dim, torch.bfloat16
    rows = gemv_tile_rows(s, b)
    order = ops.rope_pair_order(s.n_q, s.n_k, s.n_v, d, device=DEV)
    ws = _bytes(max(ops._lib.load().saga_gemv_workspace_bytes(b, n, k) for n, k in (
        (s.qkv_width, s.hidden), (s.hidden, s.n_q * d), (2 * s.intermediate, s.hidden), (s.hidden, s.intermediate))))
    packed = [{"o": ops.pack_gemv_weight(w["w_o"], rows), "gu": ops.pack_gemv_weight(w["w_gu"]),
               "d": ops.pack_gemv_weight(w["w_d"], rows), "qkv": ops.pack_gemv_weight(w["w_qkv"][order].contiguous(), rows),
               "b": w["b_qkv"][order].contiguous(), "attn": w["attn"],
               "q": torch.empty(b, s.n_q, d, dtype=dt, device=DEV),
               "k": torch.zeros(b, s.n_k, PROJ_POSITIONS, d, dtype=dt, device=DEV),
               "v": torch.zeros(b, s.n_v, PROJ_POSITIONS, d, dtype=dt, device=DEV)} for w in layers]
    x, act = torch.empty_like(x0), torch.empty(b, s.intermediate, dtype=dt, device=DEV)
    table = ops.rope_table(pos, d, s.rope_theta)

    def call():
        x.copy_(x0)
        for w in packed:
            ops.gemv(w["attn"], w["o"], epilogue="add", out=x, workspace=ws)
            ops.gemv(x, w["gu"], rms_eps=s.eps, epilogue="silu_pairs", out=act, workspace=ws)
            ops.gemv(act, w["d"], epilogue="add", out=x, workspace=ws)
            ops.gemv_rope_kv(x, w["qkv"], w["b"], s.n_q, s.n_k, s.n_v, s.rope_theta, pos, w["k"], w["v"], rms_eps=s.eps,
                             q_out=w["q"], rope_table=table)

    outs = {"x": x, "q": [w["q"] for w in packed], "k": [w["k"] for w in packed], "v": [w["v"] for w in packed]}
    return {"graph": _graphed(call), "outs": outs, "keep": (call, ws, x0, table)}


def _value_mean(s, seed):
    """The part that a head's cached values have in common.  Without it a head's output is what is left of N(0,1)
    values averaged, and the few positions that bf16 rounding moves across the top-N cut are percents of it."""
    return _randn(_gen(seed + 2), s.layers, 1, s.n_v, 1, s.head_dim, dtype=torch.bfloat16)


def _prepare_decode(c, seed):
    s = SHAPES[c["shape"]]
    m = SagaDecoder(s, c["b"], c["L"] + 8, top_n=c["N"], weights=_weights(s, seed))
    m.fill_synthetic(c["L"], seed=seed + 1)
    m.v_cache[..., : c["L"], :] += _value_mean(s, seed)
    m.capture()
    m.tokens.fill_(1)  # the token before: its step leaves the thresholds
    m.replay(0)
    return {"model": m, "L": c["L"]}


def _prepare_prompt(c, seed):
    s = SHAPES[c["shape"]]
    m = SagaDecoder(s, 1, c["T"] + 8, top_n=512, weights=_weights(s, seed))
    return {"model": m, "prompt": torch.randint(s.vocab, (c["T"],), generator=_gen(seed + 1), device=DEV)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attn":
        s, q, k, v, mask = _attn_inputs(case, seed)
        return {"module": _Attention(), "q": q, "k": k, "v": v, "mask": mask}
    if kind == "proj":
        return _prepare_proj(case, seed)
    if kind == "decode":
        return _prepare_decode(case, seed)
    if kind == "prompt":
        return _prepare_prompt(case, seed)
    return _prepare_decode_attention(case, seed)


# --------------------------------------------------------------------- pass

@torch.no_grad()
def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    if "table" in state:
        A.AMORTIZED_THRESHOLD_TENSOR = state["table"]
        return A.approx_top_n_attention_amortized(state["q"], state["k"], state["v"], state["mask"],
                                                  top_n_attention=state["N"], layer_idx=0)
    if "module" in state:
        return A.sdpa_attention_forward(state["module"], state["q"], state["k"], state["v"], state["mask"])[0]
    m = state["model"]
    if "prompt" in state:
        # the caches are what a prompt leaves for the decode steps
        m.prefill(state["prompt"])
        return {"k": m.k_cache, "v": m.v_cache}
    m.reset()
    m.replay(1)
    at = state["L"]  # the position this step appended
    return {"logits": m._logits, "k": m.k_cache[..., at, :], "v": m.v_cache[..., at, :]}


# --------------------------------------------------------------------- work

def _layer_weights(s):
    return s.qkv_width * s.hidden + s.hidden * s.n_q * s.head_dim + 3 * s.intermediate * s.hidden


def work(case):
    c, s, kind = case, SHAPES[case["shape"]], case["kind"]
    d = s.head_dim
    if kind == "prompt":
        T = c["T"]
        flops = s.layers * (2 * T * _layer_weights(s) + 2 * s.n_q * d * T * (T + 1)) + 2 * s.vocab * s.hidden
        kv = s.layers * (s.n_k + s.n_v) * T * d * 2
        return {"bytes": 2 * (s.layers * _layer_weights(s) + s.vocab * s.hidden) + kv, "flops": flops}
    if kind == "proj":
        w = PROJ_LAYERS * _layer_weights(s)
        io = 2 * c["b"] * (2 * s.hidden + PROJ_LAYERS * (s.n_q * d + s.qkv_width))
        return {"bytes": 2 * w + io, "flops": 2 * c["b"] * w}
    if kind == "attn":
        pairs = sum((c["T"] - p) * (c["T"] - p + 1) // 2 for p in (_pads(c) if c["masked"] else [0] * c["b"]))
        io = 2 * c["b"] * c["T"] * d * (2 * s.n_q + s.n_k + s.n_v) + (c["b"] * c["T"] ** 2 if c["masked"] else 0)
        return {"bytes": io, "flops": 4 * s.n_q * d * pairs}
    if kind == "decode":
        w = s.layers * _layer_weights(s) + s.vocab * s.hidden
        att, ops_ = _attention_work(s, [c["L"] + 1] * c["b"], c["N"])
        return {"bytes": 2 * w + s.layers * att + 2 * c["b"] * s.vocab, "flops": 2 * c["b"] * w + s.layers * ops_}
    n, f = _attention_work(s, _kv_lens(c), None if kind == "dense" else c["N"])
    return {"bytes": n + (2 * c["b"] * c["L"] if c.get("mask") else 0), "flops": f}


def _attention_work(s, lens, N):
    """One decode attention call: keys, the value rows that a head keeps (all of them: dense), q and out."""
    d, n, f = s.head_dim, 0, 0
    for L in lens:
        kept = L if N is None else min(N, L)
        n += 2 * d * (s.n_k * L + min(s.n_v * L, s.n_q * kept) + 2 * s.n_q) + (4 * s.n_q if N is not None else 0)
        f += 2 * s.n_q * d * (L + kept)
    return n, f


def tolerance(case):
    """About four times the distance from 64 bits, measured over the listed and drawn cases: bf16 outputs 1.6e-3 to
    2.2e-3, f16 2e-4 to 3e-4 (a position at the cut of a fast step may fall either way: same bound in both types), the
    chains of bf16 roundings in "proj" 4.6e-3; "decode" and "prompt" round the residual stream twice a layer, 1e-2 to
    2.4e-2 at the last of 28 or 32."""
    kind, f16 = case["kind"], case.get("dtype") == "f16"
    if kind in ("calibrate", "dense", "attn"):
        return {"rel": 1.2e-3 if f16 else 8e-3}
    return {"rel": {"call": 8e-3, "atopn": 8e-3, "proj": 1.6e-2, "decode": 3e-2, "prompt": 3e-2}[kind]}


# -------------------------------------------------------- the same in 64 bits

def _logits64(q, k, mask, i, n, scale=None):
    """Logits [q_h, n] of batch row i over its first n positions."""
    q_h, d, k_h = q.shape[1], q.shape[3], k.shape[1]
    x = torch.matmul(q[i].double().reshape(k_h, q_h // k_h, d), k[i, :, :n].double().transpose(1, 2)).reshape(q_h, n)
    x = x * (1 / math.sqrt(d))
    return x if mask is None else x + mask[i, :, 0, :n].double()


def _weights64(x, N, pstar, cal):
    """Attention weights [q_h, n] of logits x: dense, the exact top N (cal), or the positions above p*'s logit; and
    the N-th largest probability."""
    if N is None:
        return torch.softmax(x, dim=-1), None
    if cal:
        p = torch.softmax(x, dim=-1)
        top = p.topk(min(N, x.shape[1]), dim=-1)
        kept = torch.zeros_like(p).scatter_(1, top.indices, top.values)
        return kept / kept.sum(-1, keepdim=True), top.values[:, -1]
    m = x[:, -256:].max(dim=-1, keepdim=True).values
    t = m + torch.log(pstar.double().clamp(min=1e-30)[:, None] * torch.exp(x - m).sum(-1, keepdim=True))
    keep = x > t
    keep &= keep.cumsum(-1) <= min(2 * N, x.shape[1])  # at most 2 N of them, in order of position
    return torch.softmax(x.masked_fill(~keep, -math.inf), dim=-1), None


def _times_v64(p, v, i, n):
    q_h, v_h = p.shape[0], v.shape[1]
    return torch.matmul(p.reshape(v_h, q_h // v_h, n), v[i, :, :n].double()).reshape(q_h, v.shape[3])


def _attention64(q, k, v, lens, mask, N, pstar, cal):
    out, thr = [], []
    q_h = q.shape[1]
    for i, n in enumerate(lens):
        p, t = _weights64(_logits64(q, k, mask, i, n), N, None if pstar is None else pstar[i * q_h:(i + 1) * q_h], cal)
        out.append(_times_v64(p, v, i, n))
        thr.append(t)
    return torch.stack(out)[:, :, None], (torch.cat(thr) if cal else None)


def _norm64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, pos, theta):
    """Rotate-half on x [T, heads, d]."""
    h = x.shape[-1] // 2
    a = pos.double()[:, None] * theta ** (-torch.arange(h, device=DEV, dtype=torch.float64) / h)[None, :]
    co, si = a.cos()[:, None], a.sin()[:, None]
    return torch.cat([x[..., :h] * co - x[..., h:] * si, x[..., h:] * co + x[..., :h] * si], dim=-1)


def _mlp64(s, x, w_gu, w_d, ln):
    gu = _norm64(x, ln, s.eps) @ w_gu.double().t()
    return x + (torch.nn.functional.silu(gu[:, :s.intermediate]) * gu[:, s.intermediate:]) @ w_d.double().t()


def _qkv64(s, x, w, bias, ln, pos):
    qkv = (_norm64(x, ln, s.eps) @ w.double().t() + bias.double()).reshape(x.shape[0], -1, s.head_dim)
    q, k, v = qkv.split([s.n_q, s.n_k, s.n_v], dim=1)
    return _rope64(q, pos, s.rope_theta), _rope64(k, pos, s.rope_theta), v


def _causal64(q, k, v, pad=0):
    """q [q_h, T, d] over k, v [h, T, d]: causal, the first `pad` keys hidden; blocks of queries keep it small."""
    q_h, T, d = q.shape
    k, v = (x.repeat_interleave(q_h // x.shape[0], 0).double() for x in (k, v))
    out, ar = [], torch.arange(T, device=DEV)
    for i in range(0, T, 512):
        x = torch.matmul(q[:, i:i + 512].double(), k.transpose(1, 2)) / math.sqrt(d)
        keep = (ar[None, :] <= ar[i:i + 512, None]) & (ar[None, :] >= pad)
        p = torch.softmax(x.masked_fill(~keep, -math.inf), dim=-1)
        out.append(torch.matmul(p.nan_to_num(0.0), v))  # a query that sees no key gives 0
    return torch.cat(out, dim=1)


def _exact_proj(c, seed):
    s, x, layers, pos = _proj_inputs(c, seed)
    x, one, b = x.double(), torch.ones(s.hidden, device=DEV), c["b"]
    outs = {"q": [], "k": [], "v": []}
    for w in layers:
        x = x + w["attn"].double() @ w["w_o"].double().t()
        x = _mlp64(s, x, torch.cat([w["w_gu"][0::2], w["w_gu"][1::2]]), w["w_d"], one)
        q, k, v = _qkv64(s, x, w["w_qkv"], w["b_qkv"], one, pos)
        outs["q"].append(q)
        for name, new in (("k", k), ("v", v)):
            cache = torch.zeros(b, new.shape[1], PROJ_POSITIONS, s.head_dim, dtype=torch.float64, device=DEV)
            cache[torch.arange(b, device=DEV), :, pos.long()] = new
            outs[name].append(cache)
    return {"x": x, **outs}


def _exact_decode(c, seed):
    s, b, L = SHAPES[c["shape"]], c["b"], c["L"]
    w, g = _weights(s, seed), _gen(seed + 1)
    # the cache contents of SagaDecoder.fill_synthetic
    k_all, v_all = (torch.randn(s.layers, b, h, L, s.head_dim, generator=g, device=DEV).to(torch.bfloat16)
                    for h in (s.n_k, s.n_v))
    v_all += _value_mean(s, seed)
    pos, pstar = torch.full((b,), L, device=DEV), [None] * s.layers
    for token, cal in ((1, True), (0, False)):
        x, ks, vs = w["embed"][token].double().expand(b, -1), [], []
        for l in range(s.layers):
            q, k, v = _qkv64(s, x, w["w_qkv"][l], w["b_qkv"][l], w["ln1"][l], pos)
            ks.append(k)
            vs.append(v)
            k1 = torch.cat([k_all[l].double(), k[:, :, None]], dim=2)
            v1 = torch.cat([v_all[l].double(), v[:, :, None]], dim=2)
            o, t = _attention64(q[:, :, None], k1, v1, [L + 1] * b, None, c["N"], pstar[l], cal)
            pstar[l] = t
            x = x + o.reshape(b, -1) @ w["w_o"][l].double().t()
            x = _mlp64(s, x, w["w_gu"][l], w["w_d"][l], w["ln2"][l])
    logits = _norm64(x, w["ln_f"], s.eps) @ w["embed"].double().t()
    return {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs)}


def _exact_prompt(c, seed):
    s, T = SHAPES[c["shape"]], c["T"]
    w = _weights(s, seed)
    x = w["embed"][torch.randint(s.vocab, (T,), generator=_gen(seed + 1), device=DEV)].double()
    kc, vc = (torch.zeros(s.layers, 1, h, T + 8, s.head_dim, dtype=torch.float64, device=DEV) for h in (s.n_k, s.n_v))
    pos = torch.arange(T, device=DEV)
    for l in range(s.layers):
        q, k, v = _qkv64(s, x, w["w_qkv"][l], w["b_qkv"][l], w["ln1"][l], pos)
        kc[l, 0, :, :T], vc[l, 0, :, :T] = k.transpose(0, 1), v.transpose(0, 1)
        if l + 1 < s.layers:  # the last layer's output reaches no cache
            o = _causal64(q.transpose(0, 1), kc[l, 0, :, :T], vc[l, 0, :, :T])
            x = x + o.transpose(0, 1).reshape(T, -1) @ w["w_o"][l].double().t()
            x = _mlp64(s, x, w["w_gu"][l], w["w_d"][l], w["ln2"][l])
    return {"k": kc, "v": vc}


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "proj":
        return _exact_proj(c, seed)
    if kind == "decode":
        return _exact_decode(c, seed)
    if kind == "prompt":
        return _exact_prompt(c, seed)
    if kind == "attn":
        s, q, k, v, _ = _attn_inputs(c, seed)
        pads = _pads(c) if c["masked"] else [0] * c["b"]
        return torch.stack([_causal64(q[i], k[i], v[i], pads[i]).transpose(0, 1) for i in range(c["b"])])
    s, q, k, v, lens, mask, pstar = _decode_inputs(c, seed)
    out, thr = _attention64(q, k, v, lens, mask, c.get("N"), pstar, kind == "calibrate")
    return {"out": out, "thr": thr} if kind == "calibrate" else {"out": out} if kind != "call" else out
