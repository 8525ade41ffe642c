"""Performance cases of the kernel layer: what programs have it do, at the sizes they do it.

`listed()` names twelve cases; `draw(rng)` gives more of the same ranges.  Every case
goes through the package's launchers (or its graph executor) on device tensors, as a
user's program does: the tile is picked once for a shape, buffers and workspaces are
kept, and a pass is the launch itself.

Families and their ranges (odd sizes among the drawn ones):

  gemm_f32    C = alpha A B + beta C in fp32; M, N, K from 1 row up to 4096
  gemm_fused  y = act(x W + b) in one launch: the layer of an MLP over M tokens
  gemm_lp     bf16 / fp16 inputs, fp32 accumulation, fp32 or 16-bit output
  reduce      row sum / max / mean, one pass per row, or the split form (full sum)
  softmax     row softmax, one pass
  bias_act    act(x + bias)
  block       GEMM -> GELU -> GEMM -> softmax through the graph executor
"""
from __future__ import annotations

import math

import numpy as np
import torch

from __graft_entry__ import load_package

ACTS = ("none", "relu", "gelu_erf", "gelu_tanh")
KINDS = ("sum", "max", "mean")
MAX_GEMM_FLOPS = 2 * 4096 ** 3
MAX_ELEMENTS = 1 << 27


def listed():
    return [
        # The smallest square product of the benchmark's sweep: one short launch.
        {"name": "gemm_f32_512", "op": "gemm_f32", "m": 512, "n": 512, "k": 512,
         "alpha": 1.0, "beta": 0.0},
        # An ordinary large product, whole tiles.
        {"name": "gemm_f32_4096", "op": "gemm_f32", "m": 4096, "n": 4096, "k": 4096,
         "alpha": 1.0, "beta": 0.0},
        # Odd in every extent, accumulated into C: a solver's or a statistics program's
        # matrix, whose sizes come from its data.
        {"name": "gemm_f32_odd", "op": "gemm_f32", "m": 1531, "n": 1021, "k": 2053,
         "alpha": 0.5, "beta": 1.5},
        # A few rows through a wide layer: a small batch, bound by reading the weights.
        {"name": "gemm_f32_few_rows", "op": "gemm_f32", "m": 16, "n": 4096, "k": 4096,
         "alpha": 1.0, "beta": 0.0},
        # The first layer of an MLP over a batch whose token count is not a tile multiple.
        {"name": "fused_tokens", "op": "gemm_fused", "m": 3000, "n": 4096, "k": 1024,
         "act": "gelu_tanh"},
        # 16-bit training or prefill product, whole tiles.
        {"name": "gemm_bf16_4096", "op": "gemm_lp", "m": 4096, "n": 4096, "k": 4096,
         "ab": "bf16", "c": "bf16"},
        # 16-bit layer over a ragged batch, fp32 output.
        {"name": "gemm_f16_tokens", "op": "gemm_lp", "m": 1531, "n": 4096, "k": 1024,
         "ab": "f16", "c": "f32"},
        # Means of many short rows: per-sample or per-head statistics.
        {"name": "row_mean_short", "op": "reduce", "kind": "mean", "variant": "shuffle",
         "rows": 131072, "cols": 200},
        # The full-tensor sum (a loss or a norm over all elements), split form.
        {"name": "full_sum", "op": "reduce", "kind": "sum", "variant": "two_pass",
         "rows": 1, "cols": 1 << 26},
        # Softmax over a vocabulary-sized row, odd width.
        {"name": "softmax_long_odd", "op": "softmax", "rows": 4096, "cols": 32001},
        # bias + GELU over rows of odd width (no vector width but 1 is legal).
        {"name": "bias_gelu_odd", "op": "bias_act", "act": "gelu_tanh", "rows": 16384,
         "cols": 4095},
        # A whole call: the transformer MLP block planned on the graph executor, its
        # output read back by the host program.
        {"name": "block_1000", "op": "block", "tokens": 1000, "d": 1024, "ff": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _extent(rng, lo, hi):
    """An extent in [lo, hi], log-uniform: a multiple of 64, a multiple of 8, or any."""
    v = _log_int(rng, lo, hi)
    step = rng.choice((64, 8, 1, 1))
    return min(hi, max(lo, v // step * step)) if v >= step else v


def draw(rng):
    op = rng.choice(("gemm_f32", "gemm_f32", "gemm_fused", "gemm_lp", "gemm_lp", "reduce",
                     "reduce", "softmax", "softmax", "bias_act", "block"))
    if op in ("gemm_f32", "gemm_fused", "gemm_lp"):
        while True:
            # One product in four has few rows (a small batch).
            m = _log_int(rng, 1, 64) if rng.random() < 0.25 else _extent(rng, 64, 4096)
            n, k = _extent(rng, 128, 8192), _extent(rng, 128, 8192)
            if 2 * m * n * k <= MAX_GEMM_FLOPS:
                break
        case = {"op": op, "m": m, "n": n, "k": k}
        if op == "gemm_f32":
            case["alpha"], case["beta"] = rng.choice(((1.0, 0.0), (1.0, 0.0), (0.5, 1.5)))
        elif op == "gemm_fused":
            case["act"] = rng.choice(ACTS)
        else:
            case["ab"] = rng.choice(("bf16", "f16"))
            case["c"] = rng.choice(("f32", case["ab"]))
        return case
    if op == "block":
        d = rng.choice((512, 768, 1024))
        return {"op": op, "tokens": _extent(rng, 128, 4096), "d": d, "ff": 4 * d}
    if op == "reduce":
        kind = rng.choice(KINDS)
        if rng.random() < 0.25:
            # A tensor reduced whole, or in a few long pieces.
            rows = rng.choice((1, 1, _log_int(rng, 1, 64)))
            cols = _extent(rng, 1 << 16, MAX_ELEMENTS // rows)
            return {"op": op, "kind": kind, "variant": "two_pass", "rows": rows, "cols": cols}
        cols = _extent(rng, 16, 32768)
        rows = _log_int(rng, 256, min(262144, MAX_ELEMENTS // cols))
        return {"op": op, "kind": kind, "variant": "shuffle", "rows": rows, "cols": cols}
    if op == "softmax":
        cols = _extent(rng, 32, 65536)
        return {"op": op, "rows": _log_int(rng, 256, min(65536, MAX_ELEMENTS // cols)),
                "cols": cols}
    cols = _extent(rng, 64, 16384)
    return {"op": op, "act": rng.choice(ACTS),
            "rows": _log_int(rng, 64, min(65536, (MAX_ELEMENTS // 2) // cols)), "cols": cols}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(g, shape, lo, hi):
    return torch.empty(shape, device="cuda", dtype=torch.float32).uniform_(lo, hi, generator=g)


def _normal(g, shape, sigma):
    return torch.empty(shape, device="cuda", dtype=torch.float32).normal_(0.0, sigma, generator=g)


def _inputs(case, seed):
    """The case's input tensors, from the seed alone."""
    g = _gen(seed)
    op = case["op"]
    if op == "gemm_f32":
        m, n, k = case["m"], case["n"], case["k"]
        return {"a": _uniform(g, (m, k), -1.0, 1.0), "b": _uniform(g, (k, n), -1.0, 1.0),
                "c": _uniform(g, (m, n), -1.0, 1.0)}
    if op == "gemm_fused":
        m, n, k = case["m"], case["n"], case["k"]
        return {"a": _normal(g, (m, k), 1.0), "b": _normal(g, (k, n), 1.0 / math.sqrt(k)),
                "bias": _normal(g, (n,), 0.1)}
    if op == "gemm_lp":
        m, n, k = case["m"], case["n"], case["k"]
        t = _TORCH[case["ab"]]
        return {"a": _normal(g, (m, k), 1.0).to(t),
                "b": _normal(g, (k, n), 1.0 / math.sqrt(k)).to(t)}
    if op == "reduce":
        return {"x": _uniform(g, (case["rows"], case["cols"]), 0.0, 1.0)}
    if op == "softmax":
        # Logits N(0, 2^2), one row in a hundred with a spike.
        x = _normal(g, (case["rows"], case["cols"]), 2.0)
        rows = max(1, case["rows"] // 100)
        x[:rows, case["cols"] // 3] += 30.0
        return {"x": x}
    if op == "bias_act":
        return {"x": _normal(g, (case["rows"], case["cols"]), 1.0),
                "bias": _uniform(g, (case["cols"],), -0.5, 0.5)}
    tokens, d, ff = case["tokens"], case["d"], case["ff"]
    return {"x": _normal(g, (tokens, d), 1.0), "w1": _normal(g, (d, ff), 1.0 / math.sqrt(d)),
            "b1": _normal(g, (ff,), 0.1), "w2": _normal(g, (ff, d), 1.0 / math.sqrt(ff))}


def prepare(case, seed):
    mcke = load_package()
    mcke.lib()
    s = {"case": case, "mcke": mcke}
    s.update(_inputs(case, seed))
    op = case["op"]
    if op == "gemm_f32":
        s["tile"] = mcke.gemm_mfma_default_tile(case["m"], case["n"], case["k"])
        s["c0"] = s["c"]
        s["c"] = s["c0"].clone()
    elif op == "gemm_fused":
        s["tile"] = mcke.gemm_mfma_default_tile(case["m"], case["n"], case["k"])
        s["y"] = torch.empty((case["m"], case["n"]), device="cuda")
        s["act"] = mcke.Activation(ACTS.index(case["act"]))
    elif op == "gemm_lp":
        kinds = {"f32": mcke.DType.kF32, "f16": mcke.DType.kF16, "bf16": mcke.DType.kBF16}
        s["tile"] = mcke.gemm_lp_default_tile(case["m"], case["n"], case["k"])
        s["ab"], s["cd"] = kinds[case["ab"]], kinds[case["c"]]
        s["c"] = torch.empty((case["m"], case["n"]), device="cuda", dtype=_TORCH[case["c"]])
    elif op == "reduce":
        s["kind"] = mcke.ReduceKind(KINDS.index(case["kind"]))
        s["out"] = torch.empty((case["rows"],), device="cuda")
        if case["variant"] == "two_pass":
            s["ws_bytes"] = mcke.row_reduce_workspace_bytes(case["rows"], case["cols"],
                                                            mcke.ReduceVariant.kTwoPass)
            s["ws"] = torch.empty((max(1, s["ws_bytes"] // 4),), device="cuda")
    elif op == "softmax":
        s["y"] = torch.empty_like(s["x"])
    elif op == "bias_act":
        s["y"] = torch.empty_like(s["x"])
        s["act"] = mcke.Activation(ACTS.index(case["act"]))
        s["vw"] = min(mcke.max_vector_width_f32(s[t], case["cols"]) for t in ("x", "y", "bias"))
    else:
        import mcke_amd.graph as mg
        g, t = mg.transformer_block_fused(case["tokens"], case["d"], case["ff"])
        ex = mg.Executor(g)
        ex.plan()
        for name, key in (("x", "x"), ("W1", "w1"), ("b1", "b1"), ("W2", "w2")):
            ex.set_input(t[name], s.pop(key).cpu().numpy())
        s["ex"], s["out"] = ex, t["softmax"]
    return s


def run(s):
    case, mcke = s["case"], s["mcke"]
    op = case["op"]
    if op == "gemm_f32":
        if case["beta"] != 0.0:
            s["c"].copy_(s["c0"])   # the matrix that this pass accumulates into
        st = mcke.launch_gemm_f32(s["a"], s["b"], s["c"], case["m"], case["n"], case["k"],
                                  case["alpha"], case["beta"], mcke.GemmVariant.kMfmaF32,
                                  s["tile"])
        out = s["c"]
    elif op == "gemm_fused":
        st = mcke.launch_gemm_bias_act_f32(s["a"], s["b"], s["bias"], s["y"], case["m"],
                                           case["n"], case["k"], 1.0, s["act"], s["tile"])
        out = s["y"]
    elif op == "gemm_lp":
        st = mcke.launch_gemm_lp(s["a"], s["b"], s["c"], s["ab"], s["cd"], case["m"], case["n"],
                                 case["k"], 1.0, 0.0, s["tile"])
        out = s["c"]
    elif op == "reduce":
        if case["variant"] == "two_pass":
            st = mcke.launch_row_reduce_f32(s["x"], s["out"], case["rows"], case["cols"],
                                            s["kind"], mcke.ReduceVariant.kTwoPass, s["ws"],
                                            s["ws_bytes"], None)
        else:
            st = mcke.launch_row_reduce_f32(s["x"], s["out"], case["rows"], case["cols"],
                                            s["kind"], mcke.ReduceVariant.kWarpShuffle)
        out = s["out"]
    elif op == "softmax":
        st = mcke.launch_row_softmax_f32(s["x"], s["y"], case["rows"], case["cols"],
                                         mcke.SoftmaxVariant.kOnlineOnePass)
        out = s["y"]
    elif op == "bias_act":
        st = mcke.launch_bias_act_f32(s["x"], s["bias"], s["y"], case["rows"], case["cols"],
                                      s["act"], s["vw"])
        out = s["y"]
    else:
        s["ex"].run_sync()
        return s["ex"].read(s["out"], case["tokens"] * case["d"]).reshape(case["tokens"],
                                                                          case["d"])
    st.throw_if_error()
    return out


def work(case):
    op = case["op"]
    if op in ("gemm_f32", "gemm_fused", "gemm_lp"):
        m, n, k = case["m"], case["n"], case["k"]
        ab = 2 if op == "gemm_lp" else 4
        c = 2 if op == "gemm_lp" and case["c"] != "f32" else 4
        # With beta the matrix accumulated into is read, too.
        reads = 1 if op == "gemm_f32" and case["beta"] != 0.0 else 0
        bias = 4 * n if op == "gemm_fused" else 0
        return {"bytes": ab * (m * k + k * n) + c * m * n * (1 + reads) + bias,
                "flops": 2 * m * n * k}
    if op == "reduce":
        return {"bytes": 4 * (case["rows"] * case["cols"] + case["rows"]), "flops": 0}
    if op == "softmax":
        return {"bytes": 8 * case["rows"] * case["cols"], "flops": 0}
    if op == "bias_act":
        return {"bytes": 4 * (2 * case["rows"] * case["cols"] + case["cols"]), "flops": 0}
    t, d, ff = case["tokens"], case["d"], case["ff"]
    return {"bytes": 4 * (2 * t * d + 2 * d * ff + ff), "flops": 4 * t * d * ff}


def tolerance(case):
    # About four times the error against 64-bit arithmetic measured over the ranges.
    op = case["op"]
    if op in ("gemm_f32", "gemm_fused"):
        return {"rel": 6e-6, "max": 1e-4}
    if op == "gemm_lp":
        # fp32 accumulation; a 16-bit output adds its own rounding.
        if case["c"] == "f32":
            return {"rel": 6e-6, "max": 1e-4}
        return {"rel": 6e-3, "max": 2e-2} if case["c"] == "bf16" else {"rel": 8e-4, "max": 3e-3}
    if op == "reduce":
        return "exact" if case["kind"] == "max" else {"rel": 1e-6, "max": 1e-5}
    if op == "softmax":
        return {"rel": 1e-6, "max": 2e-5}
    if op == "bias_act":
        # none and ReLU round once: the same bits.
        return "exact" if case["act"] in ("none", "relu") else {"rel": 5e-7, "max": 1e-5}
    return {"rel": 1e-5, "max": 2e-4}


def _act64(v, act):
    if act == "relu":
        return torch.clamp(v, min=0.0)
    if act == "gelu_erf":
        return 0.5 * v * (1.0 + torch.special.erf(v / math.sqrt(2.0)))
    if act == "gelu_tanh":
        return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))
    return v


def exact(case, seed):
    x = _inputs(case, seed)
    op = case["op"]
    if op == "gemm_f32":
        r = case["alpha"] * (x["a"].double() @ x["b"].double())
        return r + case["beta"] * x["c"].double() if case["beta"] != 0.0 else r
    if op == "gemm_fused":
        return _act64(x["a"].double() @ x["b"].double() + x["bias"].double(), case["act"])
    if op == "gemm_lp":
        return x["a"].double() @ x["b"].double()
    if op == "reduce":
        if case["kind"] == "max":
            return x["x"].amax(dim=1).double()
        s = x["x"].sum(dim=1, dtype=torch.float64)
        return s / case["cols"] if case["kind"] == "mean" else s
    if op == "softmax":
        return torch.softmax(x["x"].double(), dim=1)
    if op == "bias_act":
        return _act64(x["x"].double() + x["bias"].double(), case["act"])
    h = _act64(x["x"].double() @ x["w1"].double() + x["b1"].double(), "gelu_tanh")
    return torch.softmax(h @ x["w2"].double(), dim=1).cpu().numpy().astype(np.float64)
