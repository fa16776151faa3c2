"""Performance cases of the quantized-matmul library: what a serving program has it do, through
the public Python entry points (`mi_qmm`), from one decode row to an 8192-row prefill.

Three kinds of case:
  linear  one quantized linear layer, or a stack of them (a decode step's projections)
  mlp     dense SwiGLU MLP blocks: gate and up projections, SwiGLU, down projection
  moe     a routed-expert layer: routing, expert gate + up + SwiGLU, expert down, score-weighted
          slot sum; optionally with the layer's dense shared expert

A decode step (at most GRAPH_ROWS rows) is captured once into a graph and replayed, as a serving
loop does (and bench.py), with a few layers of distinct weights so that they come from HBM;
larger calls, and the cases that say `graph: False`, run eagerly.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mlx-serve_amd"))
import mi_qmm as mi  # noqa: E402

GRAPH_ROWS = 64
# bits and group size of the bias-less modes (one scale byte a group)
FP = {"nvfp4": (4, 16), "mxfp4": (4, 32), "mxfp8": (8, 32)}
MASK64 = (1 << 64) - 1


def linear(M, N, K, bits=4, gs=64, mode="affine", count=1, graph=False):
    return {"kind": "linear", "M": M, "N": N, "K": K, "bits": bits, "gs": gs, "mode": mode,
            "count": count, "graph": graph}


def mlp(M, hidden, inter, bits=4, gs=64, mode="affine", layers=1, graph=False):
    return {"kind": "mlp", "M": M, "hidden": hidden, "inter": inter, "bits": bits, "gs": gs,
            "mode": mode, "layers": layers, "graph": graph}


def moe(T, experts, hidden, inter, topk=8, bits=4, layers=1, shared_bits=0, skew=False,
        graph=False):
    return {"kind": "moe", "T": T, "experts": experts, "hidden": hidden, "inter": inter,
            "topk": topk, "bits": bits, "layers": layers, "shared_bits": shared_bits,
            "skew": skew, "graph": graph}


def listed():
    return [
        # one attention projection of one token, called by itself: latency of a single call
        dict(linear(1, 4096, 4096), name="q_proj_m1"),
        # single-stream decode through the MLPs of an 8B dense model, 4-bit
        dict(mlp(1, 4096, 14336, layers=4, graph=True), name="mlp_m1_q4"),
        # a few concurrent streams on 8-bit weights
        dict(mlp(5, 4096, 14336, bits=8, layers=4, graph=True), name="mlp_m5_q8"),
        # a full decode batch, 4-bit
        dict(mlp(32, 4096, 14336, layers=4, graph=True), name="mlp_m32_q4"),
        # a short prompt, or the last piece of a long one
        dict(mlp(77, 4096, 14336), name="mlp_m77_q4"),
        # one chunk of a chunked prefill
        dict(mlp(512, 4096, 14336), name="mlp_m512_q4"),
        # a checkpoint of mixed widths: a 6-bit projection over a medium prompt
        dict(linear(700, 4096, 14336, bits=6), name="down_m700_q6"),
        # a long prompt of no round length
        dict(mlp(2003, 4096, 14336), name="mlp_m2003_q4"),
        # the largest single product: 8192 rows of prefill through a down projection
        dict(linear(8192, 4096, 14336), name="down_m8192_q4"),
        # single-stream decode of a small-expert MoE model (128 experts, top 8)
        dict(moe(1, 128, 2048, 768, layers=4, graph=True), name="moe128_t1"),
        # its prefill chunk: every expert active, about 32 rows each
        dict(moe(512, 128, 2048, 768), name="moe128_t512"),
        # a decode batch of a large MoE model (256 experts, an 8-bit shared expert, 10% of the
        # tokens on 8 hot experts): 2 to 3 rows an expert
        dict(moe(64, 256, 7168, 2048, shared_bits=8, skew=True), name="moe256_t64"),
    ]


SHAPES = [(4096, 4096), (14336, 4096), (4096, 14336), (1024, 4096), (2048, 7168), (7168, 2048),
          (1536, 2048), (2048, 768)]
BLOCKS = [(4096, 14336), (7168, 2048), (2048, 768), (2048, 5632)]
BANKS = [(128, 2048, 768, 8), (256, 7168, 2048, 8), (64, 2048, 1536, 6)]


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def _format(rng):
    """(bits, gs, mode): mostly 4-bit groups of 64, as most checkpoints."""
    r = rng.random()
    if r < 0.45:
        return 4, 64, "affine"
    if r < 0.60:
        return 8, 64, "affine"
    if r < 0.70:
        return rng.choice((4, 8)), rng.choice((32, 128)), "affine"
    if r < 0.85:
        return rng.choice((2, 3, 5, 6)), 64, "affine"
    mode = rng.choice(sorted(FP))
    return FP[mode] + (mode,)


def draw(rng):
    kind = rng.choice(("linear", "linear", "mlp", "mlp", "moe"))
    if kind == "moe":
        experts, hidden, inter, topk = rng.choice(BANKS)
        T = _log_int(rng, 1, 600)
        return moe(T, experts, hidden, inter, topk, bits=8 if rng.random() < 0.15 else 4,
                   skew=rng.random() < 0.3, graph=T <= GRAPH_ROWS)
    bits, gs, mode = _format(rng)
    M = _log_int(rng, 1, 2500 if kind == "mlp" else 4096)
    if kind == "mlp":
        hidden, inter = rng.choice(BLOCKS)
        return mlp(M, hidden, inter, bits, gs, mode, graph=M <= GRAPH_ROWS)
    if rng.random() < 0.6:
        N, K = rng.choice(SHAPES)
    else:  # any width; whole groups, on 128-value boundaries as model dimensions are
        N, K = 4 * _log_int(rng, 64, 4096), 128 * _log_int(rng, 4, 112)
    return linear(M, N, K, bits, gs, mode, count=4 if M <= GRAPH_ROWS else 1,
                  graph=M <= GRAPH_ROWS)


# ------------------------------------------------------------------ inputs --
def _sub(seed, *tags):
    """A 64-bit seed of its own for each tensor."""
    v = (seed * 0x9E3779B97F4A7C15 + 0x1234567) & MASK64
    for t in tags:
        v = ((v ^ (t + 1)) * 0xBF58476D1CE4E5B9) & MASK64
        v ^= v >> 29
    return v


def _randn(shape, seed, std=1.0, dtype=torch.bfloat16):
    return mi.fill_randn(torch.empty(shape, dtype=dtype, device="cuda"), seed, 0.0, std)


def _weight(N, K, bits, gs, mode, seed, E=0):
    """Packed weight of ~N(0, 0.02) values: (w, scales, biases), [E, N, ..] for a bank."""
    lead = (E, N) if E else (N,)
    if mode == "affine":
        wq, s, b = mi.quantize(_randn((max(E, 1) * N, K), seed, 0.02), gs, bits)
        return wq.view(*lead, -1), s.view(*lead, -1), b.view(*lead, -1)
    w = _randn((N, K), seed, 0.02).float().view(N, K // gs, gs)
    amax = w.abs().amax(-1, keepdim=True).clamp_min(1e-12)
    if mode == "nvfp4":
        sc = (amax / 6.0).clamp_min(2.0 ** -9).to(torch.float8_e4m3fn)
        scale, sbytes = sc.float(), sc.view(torch.uint8)
    else:  # a power of two that puts the group's largest value in the top binade
        e = torch.floor(torch.log2(amax)) - (2 if mode == "mxfp4" else 8)
        scale, sbytes = torch.exp2(e), (e + 127).to(torch.uint8)
    v = w / scale
    if mode == "mxfp8":
        codes = v.clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        packed = codes.reshape(N, K).contiguous().view(torch.int32)
    else:
        edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device="cuda")
        codes = torch.bucketize(v.abs(), edges) + 8 * (v < 0)
        c = codes.reshape(N, K // 2, 2).to(torch.uint8)
        packed = (c[..., 0] | (c[..., 1] << 4)).contiguous().view(torch.int32)
    return packed, sbytes.reshape(N, K // gs).contiguous(), None


def _capture(step):
    """The step as a graph, after one eager run that sizes what the library keeps."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


def _inputs(case, seed):
    if case["kind"] == "linear":
        fmt = (case["bits"], case["gs"], case["mode"])
        return {"x": _randn((case["M"], case["K"]), _sub(seed, 0)),
                "w": [_weight(case["N"], case["K"], *fmt, _sub(seed, 1, i))
                      for i in range(case["count"])]}
    if case["kind"] == "mlp":
        fmt = (case["bits"], case["gs"], case["mode"])
        H, I = case["hidden"], case["inter"]
        return {"x": _randn((case["M"], H), _sub(seed, 0)),
                "w": [tuple(_weight(n, k, *fmt, _sub(seed, 1, i, j))
                            for j, (n, k) in enumerate(((I, H), (I, H), (H, I))))
                      for i in range(case["layers"])]}
    E, H, I, T = case["experts"], case["hidden"], case["inter"], case["T"]
    fmt = (case["bits"], 64, "affine")
    banks = [tuple(_weight(n, k, *fmt, _sub(seed, 1, i, j), E)
                   for j, (n, k) in enumerate(((I, H), (I, H), (H, I))))
             for i in range(case["layers"])]
    logits = _randn((case["layers"], T, E), _sub(seed, 2), 1.0, torch.float32)
    if case["skew"]:
        g = torch.Generator().manual_seed(_sub(seed, 3) & 0x7FFFFFFF)
        hot = torch.randperm(E, generator=g)[:8]
        pick = torch.rand(case["layers"], T, generator=g) < 0.1
        bump = torch.zeros(case["layers"], T, E)
        bump[:, :, hot] = 8.0
        logits += (bump * pick[..., None]).cuda()
    S = {"x": _randn((T, H), _sub(seed, 0)), "w": banks, "logits": logits}
    if case["shared_bits"]:
        f = (case["shared_bits"], 64, "affine")
        S["shared"] = tuple(_weight(n, k, *f, _sub(seed, 4, j))
                            for j, (n, k) in enumerate(((I, H), (I, H), (H, I))))
    return S


def prepare(case, seed):
    S = _inputs(case, seed)
    S["case"] = case
    if case["graph"]:
        S["graph"], S["out"] = _capture(lambda: _step(S))
    return S


# -------------------------------------------------------------------- pass --
def _mlp(x, W, gs, bits, mode):
    gate, up, down = W
    h = mi.swiglu(mi.quantized_matmul(x, *gate, True, gs, bits, mode),
                  mi.quantized_matmul(x, *up, True, gs, bits, mode))
    return mi.quantized_matmul(h, *down, True, gs, bits, mode)


def _moe(x, logits, W, k, bits):
    """One routed-expert layer as the serving program runs it: few pairs read the expert banks
    in place, more are sorted by expert."""
    G, U, D = W
    T, H = x.shape
    E = logits.shape[-1]
    if T == 1:
        act, inds, sc = mi.moe_route_gate_up_swiglu(logits, x, *G, *U, k, 64, bits)
        return mi.gather_qmv_down_reduce(act, *D, inds, sc, 64, bits), inds, sc
    inds, sc = mi.moe_route_topk(logits, k, torch.bfloat16)
    if T * k < 64:
        act = mi.gather_qmv_gate_up_swiglu(x, *G, *U, inds, 64, bits)
        return mi.gather_qmv_down_reduce(act, *D, inds, sc, 64, bits), inds, sc
    order, inv, srt, lhs, seg = mi.moe_sort_dispatch(inds.reshape(-1), k, E)
    a = mi.gather_qmm_gate_up_swiglu(x.view(T, 1, H), *G, *U, lhs_indices=lhs, rhs_indices=srt,
                                     group_size=64, bits=bits, sorted_indices=True)
    v = mi.gather_qmm(a, *D, rhs_indices=srt, group_size=64, bits=bits, sorted_indices=True)
    return mi.moe_down_reduce_rows(v.view(T * k, H), inv, sc), inds, sc


def _step(S):
    c, x = S["case"], S["x"]
    if c["kind"] == "linear":
        return [mi.quantized_matmul(x, *w, True, c["gs"], c["bits"], c["mode"]) for w in S["w"]]
    if c["kind"] == "mlp":
        return [_mlp(x, W, c["gs"], c["bits"], c["mode"]) for W in S["w"]]
    out = {"layers": [_moe(x, S["logits"][i], W, c["topk"], c["bits"])
                      for i, W in enumerate(S["w"])]}
    if c["shared_bits"]:
        out["shared"] = _mlp(x, S["shared"], 64, c["shared_bits"], "affine")
    return out


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _step(state)


# ----------------------------------------------------------- what it takes --
def _wbytes(N, K, bits, gs, mode):
    return N * K * bits // 8 + N * (K // gs) * (4 if mode == "affine" else 1)


def work(case):
    if case["kind"] == "linear":
        M, N, K, n = case["M"], case["N"], case["K"], case["count"]
        w = _wbytes(N, K, case["bits"], case["gs"], case["mode"])
        return {"bytes": n * (w + 2 * M * N) + 2 * M * K, "flops": 2 * n * M * N * K}
    if case["kind"] == "mlp":
        M, H, I, n = case["M"], case["hidden"], case["inter"], case["layers"]
        f = (case["bits"], case["gs"], case["mode"])
        return {"bytes": n * (2 * _wbytes(I, H, *f) + _wbytes(H, I, *f) + 2 * M * H) + 2 * M * H,
                "flops": n * 6 * M * H * I}
    T, E, H, I, k, n = (case[f] for f in ("T", "experts", "hidden", "inter", "topk", "layers"))
    distinct = E * (1.0 - (1.0 - k / E) ** T)
    per = 3 * _wbytes(I, H, case["bits"], 64, "affine")
    byts = n * (distinct * per + 4 * T * E + 2 * T * H + 6 * T * k) + 2 * T * H
    flops = n * 6 * T * k * H * I
    if case["shared_bits"]:
        byts += 3 * _wbytes(I, H, case["shared_bits"], 64, "affine") + 2 * T * H
        flops += 6 * T * H * I
    return {"bytes": int(byts), "flops": flops}


def tolerance(case):
    # One bf16 rounding of an fp32 sum, and on some routes of the weights: two right results
    # differ by about 2.5e-3 (relative, 2-norm); a block adds the roundings of its
    # intermediates (3e-3 for an MLP, 5e-3 through the bf16 slot sum of a MoE layer).
    if case["kind"] == "linear":
        return {"rel": 0.01}
    return {"rel": 0.012 if case["kind"] == "mlp" else 0.015, "differ": 0.0}


# ---------------------------------------------------------- 64-bit results --
def _e4m3(b):
    """fp64 values of e4m3 bytes, with 0x7F / 0xFF as +-480 (these weights hold neither)."""
    b = b.to(torch.int64)
    e, m = (b >> 3) & 15, (b & 7).double()
    v = torch.where(e == 0, m * 2.0 ** -9, (1 + m / 8) * torch.exp2(e.double() - 7))
    return torch.where(b >= 128, -v, v)


def _dense(W, bits, gs, mode):
    """The fp64 matrix that a packed weight stands for."""
    w, s, b = W
    N = w.shape[0]
    K = w.shape[1] * 32 // bits
    u = w.to(torch.int64) & 0xFFFFFFFF
    u = u.view(N, K // 32, bits)  # 32 codes are `bits` dwords, lowest bits first
    cols = []
    for j in range(32):
        i, o = divmod(j * bits, 32)
        v = u[..., i] >> o
        if o + bits > 32:
            v = v | (u[..., i + 1] << (32 - o))
        cols.append((v & ((1 << bits) - 1)).to(torch.uint8))
    q = torch.stack(cols, -1).view(N, K // gs, gs)
    if mode == "affine":
        return (q.double() * s.double()[..., None] + b.double()[..., None]).view(N, K)
    if mode == "mxfp8":
        v = _e4m3(q)
    else:
        table = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device="cuda")
        v = table[(q & 7).long()] * torch.where(q >= 8, -1.0, 1.0).double()
    sc = _e4m3(s) if mode == "nvfp4" else torch.exp2(s.double() - 127)
    return (v * sc[..., None]).view(N, K)


def _swiglu64(g, u):
    return g * torch.sigmoid(g) * u


def _mlp64(x, W, bits, gs, mode):
    gate, up, down = W
    h = _swiglu64(x @ _dense(gate, bits, gs, mode).T, x @ _dense(up, bits, gs, mode).T)
    return h @ _dense(down, bits, gs, mode).T


def exact(case, seed):
    S = _inputs(case, seed)
    x = S["x"].double()
    if case["kind"] == "linear":
        return [x @ _dense(w, case["bits"], case["gs"], case["mode"]).T for w in S["w"]]
    if case["kind"] == "mlp":
        return [_mlp64(x, W, case["bits"], case["gs"], case["mode"]) for W in S["w"]]
    k, bits, layers = case["topk"], case["bits"], []
    for i, (G, U, D) in enumerate(S["w"]):
        top = torch.topk(S["logits"][i].double(), k, dim=-1)
        p = torch.softmax(top.values, -1)
        y = torch.zeros_like(x)
        for e in torch.unique(top.indices).tolist():
            t, slot = torch.nonzero(top.indices == e, as_tuple=True)
            one = [tuple(m[e] for m in bank) for bank in (G, U, D)]
            y.index_add_(0, t, _mlp64(x[t], one, bits, 64, "affine") * p[t, slot][:, None])
        layers.append((y, None, p))
    out = {"layers": layers}
    if case["shared_bits"]:
        out["shared"] = _mlp64(x, S["shared"], case["shared_bits"], 64, "affine")
    return out
