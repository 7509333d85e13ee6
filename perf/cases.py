"""The work that programs have this backend do, as cases to be timed and checked.

A case is a dict of plain values; its "op" says which of the functions below
prepares it, runs it through the C ABI's Python binding (train.cpp_amd/hip.py)
and forms its exact result:

  qmatvec    y = W x with W in a GGUF legacy quant format, the layer call of a
             decode step (one column per sequence) or of a short prompt
  dequant    one quantized tensor to F32, the work of a GGUF warm start
  prefill    a quantized weight against more columns than the fused product
             takes: dequantized to scratch, then the F32 product, the two calls
             graph_compute makes for such a node
  linear     y = W x in F32 at decode or short-prompt size (the layer call after
             a warm start)
  step       one training step of a Linear layer with bias under the squared
             loss: the calls graph_compute makes for the graph autograd builds
             (accumulators cleared, forward, loss, gradients of W, x and b)
  attention  grouped-query scores, their scaling, the product with the values
             and the copy that merges the heads (the permuted and transposed
             views and the plane broadcast of ggml graphs)
  scores_bwd the backward of one batched, broadcast product: both operands'
             gradients, the transposed copy and the sum over broadcast planes
"""
import importlib.util
import math
import sys
from pathlib import Path

import torch


def _package():
    """This repository's package; its folder's name has a dot, so it is loaded by its file."""
    if "traincpp_amd" not in sys.modules:
        pkg = Path(__file__).resolve().parent.parent / "train.cpp_amd"
        spec = importlib.util.spec_from_file_location("traincpp_amd", pkg / "__init__.py",
                                                      submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["traincpp_amd"] = mod
        spec.loader.exec_module(mod)


_package()
from traincpp_amd import hip as H  # noqa: E402

TYPES = list(H.QUANT_TYPES)
DEVICE = "cuda"


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the MLP's up projection of a 4096-wide model at batch 1: the decode step's largest layer call
        {"name": "decode_q4_0", "op": "qmatvec", "type": "q4_0", "K": 4096, "M": 14336, "N": 1},
        # a layer of a small model at batch 1, the smallest call there is: latency and launch
        {"name": "decode_small_q8_0", "op": "qmatvec", "type": "q8_0", "K": 768, "M": 288, "N": 1},
        # eight sequences decoded together, attention-sized layer
        {"name": "batch8_q8_0", "op": "qmatvec", "type": "q8_0", "K": 4096, "M": 4096, "N": 8},
        # sixteen sequences decoded together, MLP-sized layer
        {"name": "batch16_q5_0", "op": "qmatvec", "type": "q5_0", "K": 4096, "M": 14336, "N": 16},
        # a short prompt through the MLP's down projection
        {"name": "prompt50_q4_0", "op": "qmatvec", "type": "q4_0", "K": 11008, "M": 4096, "N": 50},
        # one tensor of a warm start, in a format with mins and fifth bits
        {"name": "dequant_q5_1", "op": "dequant", "type": "q5_1", "K": 4096, "M": 11008},
        # a prompt of ordinary length through a quantized layer
        {"name": "prefill197_q4_1", "op": "prefill", "type": "q4_1", "K": 4096, "M": 14336, "N": 197},
        # a warm-started F32 layer at a decode batch
        {"name": "linear24", "op": "linear", "K": 4096, "M": 4096, "N": 24},
        # a training step of the 4096-wide Linear layer over 512 tokens
        {"name": "step_4096", "op": "step", "K": 4096, "M": 4096, "T": 512},
        # a training step of a small layer whose sizes fit no tile
        {"name": "step_ragged", "op": "step", "K": 1000, "M": 777, "T": 130},
        # four sequences of 512 new tokens over 1024 keys, 32 heads on 8 key heads
        {"name": "attention_gqa", "op": "attention", "D": 128, "TK": 1024, "TQ": 512, "HK": 8, "HQ": 32, "B": 4},
        # the gradients of a small model's scores, odd length
        {"name": "scores_bwd_odd", "op": "scores_bwd", "D": 64, "TK": 333, "TQ": 333, "HK": 4, "HQ": 12, "B": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k(rng, lo, hi):
    """A row length of a quantized tensor: blocks of 32; most models' are multiples of 256."""
    step = rng.choice([256, 256, 128, 32])
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    op = rng.choice(["qmatvec", "qmatvec", "qmatvec", "dequant", "prefill", "linear", "linear", "step", "step",
                     "attention", "scores_bwd"])
    if op == "qmatvec":
        return {"op": op, "type": rng.choice(TYPES), "K": _k(rng, 256, 14336), "M": _log(rng, 64, 16384),
                "N": rng.choice([1, 1, _log(rng, 2, 64)])}
    if op == "dequant":
        return {"op": op, "type": rng.choice(TYPES), "K": _k(rng, 256, 8192), "M": _log(rng, 64, 8192)}
    if op == "prefill":
        return {"op": op, "type": rng.choice(TYPES), "K": _k(rng, 512, 4096), "M": _log(rng, 256, 11008),
                "N": _log(rng, 65, 512)}
    if op == "linear":
        return {"op": op, "K": _log(rng, 64, 8192), "M": _log(rng, 64, 8192), "N": _log(rng, 1, 256)}
    if op == "step":
        # whole tiles, multiples of four and odd sizes
        step = rng.choice([128, 4, 1])
        return {"op": op, "K": max(step, _log(rng, 64, 4096) // step * step),
                "M": max(step, _log(rng, 64, 4096) // step * step),
                "T": max(step, _log(rng, 16, 512) // step * step)}
    hk = rng.choice([1, 2, 4, 8])
    d = rng.choice([32, 64, 80, 96, 128])
    if op == "attention":
        return {"op": op, "D": d, "TK": _log(rng, 33, 1024), "TQ": _log(rng, 1, 512), "HK": hk,
                "HQ": hk * rng.choice([1, 2, 4]), "B": rng.choice([1, 2, 4])}
    return {"op": op, "D": d, "TK": _log(rng, 33, 640), "TQ": _log(rng, 33, 512), "HK": hk,
            "HQ": hk * rng.choice([1, 3, 4]), "B": rng.choice([1, 2])}


# ------------------------------------------------------------------ inputs

def _rng(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEVICE, dtype=torch.float32) * std


def _half_bytes(g, n, lo, hi):
    v = torch.rand(n, generator=g, device=DEVICE) * (hi - lo) + lo
    return v.to(torch.float16).view(torch.uint8).reshape(n, 2)


def _blocks(g, fmt, n):
    """n blocks with the benchmark's distributions: d in [2e-4, 1e-3], m in [-0.05, 0], quants uniform."""
    parts = [_half_bytes(g, n, 2e-4, 1e-3)]
    if fmt in ("q4_1", "q5_1"):
        parts.append(_half_bytes(g, n, -0.05, 0.0))
    if fmt == "q8_0":
        q = torch.randint(-127, 128, (n, 32), generator=g, device=DEVICE, dtype=torch.int8)
        parts.append(q.view(torch.uint8))
    else:
        size = H.BLOCK_BYTES[H.QUANT_TYPES[fmt]] - 2 * len(parts)
        parts.append(torch.randint(0, 256, (n, size), generator=g, device=DEVICE, dtype=torch.uint8))
    return torch.cat(parts, 1).contiguous()


def _decode64(fmt, b):
    """The blocks' values in 64 bits, [n, 32]."""
    d = b[:, 0:2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        return b[:, 2:].contiguous().view(torch.int8).double() * d
    at = 2
    m = None
    if fmt in ("q4_1", "q5_1"):
        m = b[:, 2:4].contiguous().view(torch.float16).double()
        at = 4
    high = None
    if fmt in ("q5_0", "q5_1"):
        bits = torch.arange(8, device=b.device)
        high = ((b[:, at:at + 4, None].int() >> bits) & 1).reshape(-1, 32)
        at += 4
    qs = b[:, at:].int()
    q = torch.cat([qs & 15, qs >> 4], 1)
    if high is not None:
        q = q + 16 * high
    if m is None:
        return (q - (8 if fmt == "q4_0" else 16)).double() * d
    return q.double() * d + m


def _f32(*shape):
    return torch.empty(*shape, device=DEVICE, dtype=torch.float32)


def _t(x):
    """The ggml descriptor of a torch view: ne[0] is torch's last dimension, and a
    dimension that x does not have strides over all of x, as in ggml."""
    shape, stride = list(x.shape), list(x.stride())
    lead = 4 - x.dim()
    span = max(n * s for n, s in zip(shape, stride))
    return H.tensor(x.data_ptr(), shape[::-1] + [1] * lead, [4 * s for s in stride[::-1]] + [4 * span] * lead)


def prepare(case, seed):
    g = _rng(seed)
    H.init(0)
    c, op = case, case["op"]
    s = {"case": c, "op": op}
    if op in ("qmatvec", "dequant", "prefill"):
        K, M = c["K"], c["M"]
        s["type"] = H.QUANT_TYPES[c["type"]]
        s["w"] = _blocks(g, c["type"], K * M // 32)
        if op != "dequant":
            s["x"] = _normal(g, c["N"], K)
            s["y"] = _f32(c["N"], M)
        if op != "qmatvec":
            s["f"] = _f32(M, K)
        if op == "prefill":
            s["t"] = [_t(s["f"]), _t(s["x"]), _t(s["y"])]
    elif op == "linear":
        s["w"] = _normal(g, c["M"], c["K"], std=0.02)
        s["x"] = _normal(g, c["N"], c["K"])
        s["y"] = _f32(c["N"], c["M"])
        s["t"] = [_t(s["w"]), _t(s["x"]), _t(s["y"])]
    elif op == "step":
        K, M, T = c["K"], c["M"], c["T"]
        b = {"W": _normal(g, M, K, std=0.02), "X": _normal(g, T, K), "b": _normal(g, 1, M, std=0.1)}
        for n, shape in (("MM", (T, M)), ("Y", (T, M)), ("SQ", (T, M)), ("L", (1, 1)), ("dL", (1, 1)), ("R", (T, M)),
                         ("YR", (T, M)), ("DY", (T, M)), ("DB", (1, M)), ("DX", (T, K)), ("gW", (M, K)), ("gX", (T, K)),
                         ("gb", (1, M))):
            b[n] = _f32(*shape)
        s["b"] = b
        s["t"] = {n: _t(v) for n, v in b.items()}
        s["t"].update(Wt=_t(b["W"].t()), Xt=_t(b["X"].t()), DYt=_t(b["DY"].t()))
    elif op == "attention":
        D, TK, TQ, HK, HQ, B = (c[k] for k in ("D", "TK", "TQ", "HK", "HQ", "B"))
        s["k"] = _normal(g, B, HK, TK, D)
        s["q"] = _normal(g, B, TQ, HQ, D)          # as a projection leaves it: heads inside a token
        s["v"] = _normal(g, B, HK, TK, D)
        s["s"], s["p"] = _f32(B, HQ, TQ, TK), _f32(B, HQ, TQ, TK)
        s["o"], s["y"] = _f32(B, HQ, TQ, D), _f32(B, TQ, HQ, D)
        s["t"] = [_t(s["k"]), _t(s["q"].transpose(1, 2)), _t(s["s"]), _t(s["p"]), _t(s["v"].transpose(2, 3)),
                  _t(s["o"]), _t(s["o"].transpose(1, 2)), _t(s["y"])]
    else:
        D, TK, TQ, HK, HQ, B = (c[k] for k in ("D", "TK", "TQ", "HK", "HQ", "B"))
        a, q, dy = _normal(g, B, HK, TK, D), _normal(g, B, HQ, TQ, D), _normal(g, B, HQ, TQ, TK, std=1e-2)
        m, full, da, dq = _f32(B, HQ, D, TK), _f32(B, HQ, TK, D), _f32(B, HK, TK, D), _f32(B, HQ, TQ, D)
        s.update(a=a, q=q, dy=dy, m=m, full=full, da=da, dq=dq)
        s["t"] = [_t(dy.transpose(2, 3)), _t(q.transpose(2, 3)), _t(m), _t(m.transpose(2, 3)), _t(full), _t(da),
                  _t(a.transpose(2, 3)), _t(dy), _t(dq)]
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    op, c = s["op"], s["case"]
    if op == "qmatvec":
        K, M, N = c["K"], c["M"], c["N"]
        H.qmatvec(s["type"], s["w"].data_ptr(), K, M, K // 32 * H.BLOCK_BYTES[s["type"]], s["x"].data_ptr(), N, 4 * K,
                  s["y"].data_ptr(), 4 * M)
        return s["y"]
    if op == "dequant":
        H.dequant(s["type"], s["w"].data_ptr(), c["K"] * c["M"] // 32, s["f"].data_ptr())
        return s["f"]
    if op == "prefill":
        H.dequant(s["type"], s["w"].data_ptr(), c["K"] * c["M"] // 32, s["f"].data_ptr())
        H.mul_mat_f32(*s["t"])
        return s["y"]
    if op == "linear":
        H.mul_mat_f32(*s["t"])
        return s["y"]
    t = s["t"]
    if op == "step":
        b = s["b"]
        for n, v in (("gW", 0.0), ("gX", 0.0), ("gb", 0.0), ("dL", 1.0)):
            H.fill_f32(b[n].data_ptr(), v, b[n].numel())
        H.mul_mat_f32(t["W"], t["X"], t["MM"])
        H.add_f32(t["MM"], t["b"], t["Y"])
        H.sqr_f32(t["Y"], t["SQ"])
        H.sum_f32(t["SQ"], t["L"])
        H.repeat_f32(t["dL"], t["R"])
        H.mul_f32(t["Y"], t["R"], t["YR"])
        H.scale_f32(t["YR"], t["DY"], 2.0)
        H.repeat_back_f32(t["DY"], t["DB"])
        K, M, T = c["K"], c["M"], c["T"]
        H.acc_f32(t["gb"], t["DB"], t["gb"], 4 * M, 4 * M, 4 * M, 0, True)
        H.mul_mat_acc_f32(t["Xt"], t["DYt"], t["gW"])
        H.mul_mat_f32(t["Wt"], t["DY"], t["DX"])
        H.acc_f32(t["gX"], t["DX"], t["gX"], 4 * K, 4 * K * T, 4 * K * T, 0, True)
        return {"y": b["Y"], "loss": b["L"], "gW": b["gW"], "gX": b["gX"], "gb": b["gb"]}
    if op == "attention":
        k, q, sc, p, vt, o, om, y = t
        H.mul_mat_f32(k, q, sc)
        H.scale_f32(sc, p, c["D"] ** -0.5)
        H.mul_mat_f32(vt, p, o)
        H.cpy(om, y)
        return {"p": s["p"], "y": s["y"]}
    dyt, qt, m, mt, full, da, at, dy, dq = t
    H.mul_mat_f32(dyt, qt, m)
    H.cpy(mt, full)
    H.repeat_back_f32(full, da)
    H.mul_mat_f32(at, dy, dq)
    return {"da": s["da"], "dq": s["dq"]}


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    c, op = case, case["op"]
    if op in ("qmatvec", "dequant", "prefill"):
        K, M = c["K"], c["M"]
        w = K * M // 32 * H.BLOCK_BYTES[H.QUANT_TYPES[c["type"]]]
        if op == "dequant":
            return {"bytes": w + 4 * K * M, "flops": 2 * K * M}
        return {"bytes": w + 4 * c["N"] * (K + M), "flops": 2 * K * M * c["N"]}
    if op == "linear":
        K, M, N = c["K"], c["M"], c["N"]
        return {"bytes": 4 * (K * M + N * (K + M)), "flops": 2 * K * M * N}
    if op == "step":
        K, M, T = c["K"], c["M"], c["T"]
        # W, x and b read; y, the loss and the gradients of W, x and b written
        return {"bytes": 4 * (2 * K * M + 2 * K * T + M * T + 2 * M + 1), "flops": 6 * K * M * T}
    D, TK, TQ, HK, HQ, B = (c[k] for k in ("D", "TK", "TQ", "HK", "HQ", "B"))
    flops = 4 * D * TK * TQ * HQ * B
    if op == "attention":
        return {"bytes": 4 * B * (2 * HK * TK * D + 2 * TQ * HQ * D + HQ * TQ * TK), "flops": flops}
    return {"bytes": 4 * B * (2 * HK * TK * D + 2 * TQ * HQ * D + HQ * TQ * TK), "flops": flops}


# ------------------------------------------------------------------ results

def tolerance(case):
    """F32 results whose sums may be taken in another order: about four times the
    largest difference from exact() that these sizes showed (2.7e-7 for qmatvec,
    1.1e-6 for prefill, 1.3e-6 for step, 6e-7 for the others); dequantization
    rounds once and is bit-exact."""
    return {"qmatvec": {"rel": 1.1e-6, "max": 1.1e-5}, "dequant": "exact", "prefill": {"rel": 4.4e-6, "max": 4.4e-5},
            "linear": {"rel": 3e-6, "max": 3e-5}, "step": {"rel": 5.2e-6, "max": 5.2e-5},
            "attention": {"rel": 3e-6, "max": 3e-5}, "scores_bwd": {"rel": 3e-6, "max": 3e-5}}[case["op"]]


def exact(case, seed):
    """What run() returns, in 64 bits, from the same inputs."""
    s = prepare(case, seed)
    c, op = case, case["op"]
    if op in ("qmatvec", "dequant", "prefill"):
        w = _decode64(c["type"], s["w"]).reshape(c["M"], c["K"])
        return w if op == "dequant" else s["x"].double() @ w.t().contiguous()
    if op == "linear":
        return s["x"].double() @ s["w"].double().t().contiguous()
    if op == "step":
        W, X, b = (s["b"][n].double() for n in ("W", "X", "b"))
        Y = X @ W.t().contiguous() + b
        DY = 2 * Y
        return {"y": Y, "loss": (Y * Y).sum().reshape(1, 1), "gW": DY.t().contiguous() @ X, "gX": DY @ W,
                "gb": DY.sum(0, keepdim=True)}
    r = c["HQ"] // c["HK"]
    if op == "attention":
        k, v = (s[n].double().repeat(1, r, 1, 1) for n in ("k", "v"))  # ggml's modulo broadcast of planes
        p = s["q"].double().transpose(1, 2).contiguous() @ k.transpose(2, 3).contiguous() * c["D"] ** -0.5
        return {"p": p, "y": (p @ v).transpose(1, 2).contiguous()}
    a, q, dy = (s[n].double() for n in ("a", "q", "dy"))
    full = dy.transpose(2, 3).contiguous() @ q
    da = full.reshape(c["B"], r, c["HK"], c["TK"], c["D"]).sum(1)
    return {"da": da, "dq": dy @ a.repeat(1, r, 1, 1)}
