"""Workloads that the framework's speed is measured on.

Each case is one pass through the public entry points of ``neso_amd``: a
single attention call, a relative-position attention layer, or the linear
projections of one transformer layer.  Sizes are those of the repository's
benchmark and tests (FA2 B1 H8 N128 and B1 H16 N2048 at head_dim 64, B2 H32
N4096 causal at head_dim 128, rel-pos H8 N1500, matmuls at K = 4096,
N = 11008, W8A16 at 4096^3); ``draw`` spreads them, odd and ragged sizes
included.

Inputs are N(0, 1) activations, int4 codes uniform in [0, 15] with scales in
[0.005, 0.02], int8 weights uniform in [-128, 127], the distributions of the
repository's own benchmark inputs.
"""
from __future__ import annotations

import math

import torch

import neso_amd

F16, F32, F64 = torch.float16, torch.float32, torch.float64
DEV = "cuda"

# Decode steps (few tokens) are launch-bound, and a serving program captures
# them in a HIP graph; from this many tokens on the calls are made one by one.
GRAPH_MAX_M = 64


def listed():
    return [
        # The smallest attention call: a short prompt, where a call costs its
        # launch and its latency.
        dict(name="attn_short", kind="attn", bh=8, n=128, d=64, causal=False, dtype="f16"),
        # The ordinary attention call of an encoder layer.
        dict(name="attn_2048", kind="attn", bh=16, n=2048, d=64, causal=False, dtype="f16"),
        # Causal prefill of two long sequences at head_dim 128.
        dict(name="attn_causal_4096", kind="attn", bh=64, n=4096, d=128, causal=True, dtype="f16"),
        # fp32 Q, K, V, for a model that keeps its activations in fp32.
        dict(name="attn_f32_2048", kind="attn", bh=16, n=2048, d=64, causal=False, dtype="f32"),
        # Local attention over a long, ragged sequence, fp16 output.
        dict(name="window_ragged", kind="window", seq=4001, heads=16, d=64, left=256, right=0),
        # An encoder layer's attention with a learned relative-position table.
        dict(name="relpos_table_1500", kind="table", heads=8, n=1500, d=64, out="f32"),
        # The same with content-dependent positions: the dense bias is formed
        # from fp32 activations and used at once by the attention.
        dict(name="relpos_dense_1500", kind="dense", heads=8, n=1500, d=64),
        # One layer's seven int4 projections: one token (decode), a batch of
        # 16 tokens (decode, coarse groups) and 256 tokens (prefill).
        dict(name="w4_layer_m1", kind="w4", m=1, hidden=4096, ffn=11008, group=32),
        dict(name="w4_layer_m16", kind="w4", m=16, hidden=4096, ffn=11008, group=128),
        dict(name="w4_layer_m256", kind="w4", m=256, hidden=4096, ffn=11008, group=32),
        # One layer's seven int8 projections for a batch of eight tokens.
        dict(name="w8_layer_m8", kind="w8", m=8, hidden=4096, ffn=11008),
        # A large int8 matmul, per-channel scales.
        dict(name="w8_4096", kind="w8one", m=4096, n=4096, k=4096, scaled=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "f32", "window", "table", "dense", "w4", "w4", "w4", "w8",
                       "w8one", "w8one"])
    if kind in ("attn", "f32"):
        f32 = kind == "f32"
        d = rng.choice([32, 64, 64, 128, 128])
        n = _log_int(rng, 16, 8192)
        causal = rng.random() < 0.5
        # At most a third of the largest listed case's work (the fp32 kernels
        # run at a third of the fp16 rate).
        most = (2e10 if f32 else 9e10) / (4 * n * n * d) * (2 if causal else 1)
        if most < 1:
            n = int(n * math.sqrt(most))
        bh = min(_log_int(rng, 1, 96), max(1, int(most)))
        return dict(kind="attn", bh=bh, n=n, d=d, causal=causal, dtype="f32" if f32 else "f16")
    if kind == "window":
        seq = _log_int(rng, 64, 8192)
        d = rng.choice([32, 64, 128])
        left = _log_int(rng, 8, 1024)
        return dict(kind="window", seq=seq, heads=rng.randint(2, 24), d=d, left=left,
                    right=rng.choice([0, 0, left]))
    if kind == "table":
        n = _log_int(rng, 32, 3000)
        return dict(kind="table", heads=rng.randint(2, 24), n=n, d=rng.choice([32, 64, 64, 128]),
                    out=rng.choice(["f16", "f32"]))
    if kind == "dense":
        n = _log_int(rng, 32, 2000)
        if rng.random() < 0.5:
            n = max(32, n // 32 * 32)
        return dict(kind="dense", heads=rng.randint(2, 12), n=n, d=rng.choice([32, 64, 128]))
    if kind in ("w4", "w8"):
        hidden = 128 * rng.randint(8, 32)
        ffn = 128 * round(hidden * rng.uniform(2, 2.69) / 128)
        if kind == "w8":
            return dict(kind="w8", m=_log_int(rng, 1, 64), hidden=hidden, ffn=ffn)
        m = _log_int(rng, 1, 1024)
        while m > 256 and m * hidden * hidden > 256 * 4096 * 4096:
            m //= 2
        return dict(kind="w4", m=m, hidden=hidden, ffn=ffn, group=rng.choice([32, 32, 64, 128]))
    # One int8 matmul; a quarter of them with sizes that are no multiple of 8.
    m, n, k = (_log_int(rng, 16, 4096) for _ in range(3))
    if rng.random() < 0.25:
        while 2.0 * m * n * k > 2e9:
            m, n, k = (m + 1) // 2, n * 3 // 4, k * 3 // 4
    else:
        n, k = max(16, n // 16 * 16), max(16, k // 16 * 16)
    return dict(kind="w8one", m=m, n=n, k=k, scaled=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# Inputs

def _randn(g, *shape, dtype=F16, scale=1.0):
    x = torch.randn(shape, generator=g, device=DEV, dtype=F32)
    return (x * scale if scale != 1.0 else x).to(dtype)


def _projections(c):
    """(K, N) of one layer's projections: q, k, v, o, gate, up, down."""
    h, f = c["hidden"], c["ffn"]
    return [(h, h)] * 4 + [(h, f)] * 2 + [(f, h)]


def _w4_inputs(c, g):
    """Per projection (x [M, K], words [N, K/8], scales [N, K/group]); the
    inputs that share a tensor in the layer (q, k, v; gate, up) share it here."""
    m, group = c["m"], c["group"]
    x_attn, x_o, x_ffn = (_randn(g, m, c["hidden"]) for _ in range(3))
    x_down = _randn(g, m, c["ffn"])
    xs = [x_attn, x_attn, x_attn, x_o, x_ffn, x_ffn, x_down]
    out = []
    for (k, n), x in zip(_projections(c), xs):
        words = torch.randint(-2 ** 31, 2 ** 31, (n, k // 8), generator=g, device=DEV, dtype=torch.int32)
        scales = (torch.rand((n, k // group), generator=g, device=DEV) * 0.015 + 0.005).to(F16)
        out.append((x, words, scales))
    return out


def _w8_inputs(m, shapes, g, scaled=True):
    out = []
    for k, n in shapes:
        a = _randn(g, m, k)
        b = torch.randint(-128, 128, (k, n), generator=g, device=DEV, dtype=torch.int8)
        scale = (torch.rand((n,), generator=g, device=DEV) * 0.004 + 0.001).to(F16) if scaled else None
        out.append((a, b, scale))
    return out


def _inputs(c, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind = c["kind"]
    if kind == "attn":
        dt = F32 if c["dtype"] == "f32" else F16
        return [_randn(g, c["bh"], c["n"], c["d"], dtype=dt) for _ in range(3)]
    if kind == "window":
        return [_randn(g, c["seq"], c["heads"], c["d"]) for _ in range(3)]
    if kind == "table":
        qkv = [_randn(g, c["heads"], c["n"], c["d"]) for _ in range(3)]
        return qkv + [_randn(g, c["heads"], 2 * c["n"] - 1, dtype=F32, scale=0.5)]
    if kind == "dense":
        h, n, d = c["heads"], c["n"], c["d"]
        return [_randn(g, h, n, d, dtype=F32, scale=0.5),          # Q
                _randn(g, h, 2 * n - 1, d, dtype=F32, scale=0.5),  # K_rel
                _randn(g, h, d, dtype=F32, scale=0.1),             # bias_u
                _randn(g, h, d, dtype=F32, scale=0.1),             # bias_v
                _randn(g, h, n, d, scale=0.5),                     # K
                _randn(g, h, n, d, scale=0.5)]                     # V
    if kind == "w4":
        return _w4_inputs(c, g)
    if kind == "w8":
        return _w8_inputs(c["m"], _projections(c), g)
    return _w8_inputs(c["m"], [(c["k"], c["n"])], g, c["scaled"])


# ---------------------------------------------------------------------------
# One pass

def _w4_pass(case, inputs, outs):
    for (x, words, scales), out in zip(inputs, outs):
        neso_amd.w4a16_linear(x, words, scales, group_size=case["group"], out=out)


def _w8_pass(case, inputs, outs):
    for (a, b, scale), out in zip(inputs, outs):
        m, k = a.shape
        n = b.shape[1]
        if scale is None:
            neso_amd.w8a16_matmul(a, b, out, k, k, n, n, M=m, N=n)
        else:
            neso_amd.w8a16_scaled_matmul(a, b, out, scale, k, k, n, n, M=m, N=n)


def prepare(case, seed):
    inputs = _inputs(case, seed)
    state = dict(case=case, inputs=inputs)
    kind = case["kind"]
    if kind in ("w4", "w8", "w8one"):
        one = _w4_pass if kind == "w4" else _w8_pass
        if kind == "w4":
            outs = [torch.empty((x.shape[0], w.shape[0]), dtype=F16, device=DEV) for x, w, _ in inputs]
        else:
            outs = [torch.empty((a.shape[0], b.shape[1]), dtype=F32, device=DEV) for a, b, _ in inputs]
        state.update(outs=outs, one=one)
        if kind != "w8one" and case["m"] <= GRAPH_MAX_M:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                one(case, inputs, outs)
            state["graph"] = graph
    return state


def run(state):
    c, inputs = state["case"], state["inputs"]
    kind = c["kind"]
    if kind == "attn":
        return neso_amd.attention(*inputs, causal=c["causal"])
    if kind == "window":
        return neso_amd.window_attention(*inputs, c["left"], c["right"])
    if kind == "table":
        return neso_amd.rel_pos_attention(*inputs, out_dtype=F16 if c["out"] == "f16" else F32)
    if kind == "dense":
        q, k_rel, bias_u, bias_v, k, v = inputs
        h, n, d = q.shape
        q_u, rel_bias = neso_amd.precompute_bias_and_qu(q, k_rel, bias_u, bias_v)
        o = torch.empty((h, n, d), dtype=F16, device=DEV)
        neso_amd.rel_pos_fa2_fwd(q_u, k, v, rel_bias, o, n, d, 1.0 / math.sqrt(d), n * d, n * n, num_heads=h)
        return dict(o=o, q_u=q_u, rel_bias=rel_bias)
    if "graph" in state:
        state["graph"].replay()
    else:
        state["one"](c, inputs, state["outs"])
    return state["outs"]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how closely results agree

def _window_pairs(n, left, right):
    """Visible (query, key) pairs of a window over n positions."""
    left, right = min(left, n - 1), min(right, n - 1)
    return n * (left + right + 1) - left * (left + 1) // 2 - right * (right + 1) // 2


def work(case):
    kind = case["kind"]
    if kind == "attn":
        bh, n, d = case["bh"], case["n"], case["d"]
        pairs = n * (n + 1) // 2 if case["causal"] else n * n
        return dict(bytes=bh * n * d * (3 * (4 if case["dtype"] == "f32" else 2) + 4), flops=4 * bh * pairs * d)
    if kind == "window":
        n, h, d = case["seq"], case["heads"], case["d"]
        return dict(bytes=n * h * d * 8, flops=4 * h * d * _window_pairs(n, case["left"], case["right"]))
    if kind == "table":
        h, n, d = case["heads"], case["n"], case["d"]
        return dict(bytes=h * n * d * (6 + (2 if case["out"] == "f16" else 4)) + h * (2 * n - 1) * 4,
                    flops=4 * h * n * n * d)
    if kind == "dense":
        h, n, d = case["heads"], case["n"], case["d"]
        # fp32 Q and K_rel, fp16 K and V in; fp16 Q_u, rel_bias and O out.
        return dict(bytes=h * (4 * n * d + 4 * (2 * n - 1) * d + 4 * n * d + 2 * n * n + 4 * n * d),
                    flops=6 * h * n * n * d)
    m = case["m"]
    if kind == "w4":
        h, f = case["hidden"], case["ffn"]
        weights = sum(k * n for k, n in _projections(case))
        reads = m * (3 * h + f) * 2 + weights // 2 + weights // case["group"] * 2
        return dict(bytes=reads + m * sum(n for _, n in _projections(case)) * 2, flops=2 * m * weights)
    shapes = _projections(case) if kind == "w8" else [(case["k"], case["n"])]
    return dict(bytes=sum(2 * m * k + k * n + 2 * n + 4 * m * n for k, n in shapes),
                flops=sum(2 * m * k * n for k, n in shapes))


def tolerance(case):
    """About four times the difference of two correct implementations, from
    the error of one against 64 bits (stated beside each)."""
    kind = case["kind"]
    if kind == "attn" and case["dtype"] == "f32":
        return dict(rel=4e-6, max=4e-4)   # fp32-class products and sums: 4.4e-7
    if kind in ("attn", "window", "table", "dense"):
        return dict(rel=1.5e-3, max=0.06)  # fp16 inputs, probabilities, results: 1.3e-4 to 3e-4
    if kind == "w4":
        return dict(rel=1.5e-3, max=2e-2)  # weights and results rounded to fp16: 2.1e-4 to 2.8e-4
    return dict(rel=5e-6, max=2e-4)       # exact fp16 x int8 products, fp32 sums: 4e-7 to 7e-7


# ---------------------------------------------------------------------------
# The same results in 64 bits

def _softmax_rows(s, v):
    return torch.matmul(torch.softmax(s, dim=-1), v)


def _exact_attention(c, inputs):
    kind = c["kind"]
    table = None
    if kind == "window":
        q, k, v = (x.transpose(0, 1) for x in inputs)
    elif kind == "table":
        q, k, v, table = inputs
    else:
        q, k, v = inputs
    heads, n, d = q.shape
    out = torch.empty((heads, n, d), dtype=F64, device=DEV)
    at = torch.arange(n, device=DEV)
    diff = at[:, None] - at[None, :]  # i - j
    hidden = None
    if kind == "attn" and c["causal"]:
        hidden = diff < 0
    elif kind == "window":
        hidden = (diff > c["left"]) | (diff < -c["right"])
    for h in range(heads):
        s = torch.matmul(q[h].double(), k[h].double().t().contiguous()) / math.sqrt(d)
        if table is not None:
            s += table[h].double()[diff + n - 1]
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        out[h] = _softmax_rows(s, v[h].double())
    return out.transpose(0, 1).contiguous() if kind == "window" else out


def _exact_dense(inputs):
    q, k_rel, bias_u, bias_v, k, v = (x.double() for x in inputs)
    heads, n, d = q.shape
    q_u = q + bias_u[:, None, :]
    rel_bias = torch.empty((heads, n, n), dtype=F64, device=DEV)
    o = torch.empty((heads, n, d), dtype=F64, device=DEV)
    for h in range(heads):
        # Row i of the bias is the slice [T-1-i, 2T-1-i) of row i of this product.
        g = torch.matmul(q[h] + bias_v[h], k_rel[h].t().contiguous()).contiguous()
        rel_bias[h] = g.as_strided((n, n), (2 * n - 2, 1), n - 1)
        s = (torch.matmul(q_u[h], k[h].t().contiguous()) + rel_bias[h]) / math.sqrt(d)
        o[h] = _softmax_rows(s, v[h])
    return dict(o=o, q_u=q_u, rel_bias=rel_bias)


def _exact_w4(x, words, scales, group):
    n = words.shape[0]
    shifts = torch.arange(0, 32, 4, device=DEV, dtype=torch.int32)
    codes = ((words[:, :, None] >> shifts) & 15).reshape(n, -1, group).double()
    w = ((codes - 8) * scales.double()[:, :, None]).reshape(n, -1)
    return torch.matmul(x.double(), w.t().contiguous())


def exact(case, seed):
    inputs = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("attn", "window", "table"):
        return _exact_attention(case, inputs)
    if kind == "dense":
        return _exact_dense(inputs)
    if kind == "w4":
        return [_exact_w4(x, w, s, case["group"]) for x, w, s in inputs]
    out = []
    for a, b, scale in inputs:
        c = torch.matmul(a.double(), b.double())
        out.append(c if scale is None else c * scale.double())
    return out
