"""Performance cases of the fp32 matrix-multiplication path, through its public entry points.

Each kind of case is one piece of work that a program on this framework has it do:

  matmul        NnClGlob.Bmm of two matrices: the plain product of the Tensor API
  square_train  NnClGlob.Bmm and bmm_backward of one large product (forward, dA, dB)
  attention     the two batched products of an attention block and their backward
  linear_train  autograd.linear forward and backward (y, dx, dw, db) on a batch of sequences
  decode        one or a few rows times a weight matrix, stored [K, N] (NnClGlob.gemm) or
                [N, K] (layers.Linear), as in serving
  lstm_step     the gate product of one step of the stateful LSTM (NnClGlob.LstmHidGates)
  lstm_train    the GEMM stages of LSTM training: X W + b, dX, and dW, dU, db accumulated
  permute       NnClGlob.Permute (materialised head split, transposes)
  sum           NnClGlob.Sum over one axis

Values: uniform or normal activations, weights U(-1/sqrt(fan in), 1/sqrt(fan in)), a row
softmax for attention probabilities.
"""
import math

import numpy as np
import torch

from my_pytchon_opencl_lib_amd import NnClGlob
from my_pytchon_opencl_lib_amd.autograd import linear
from my_pytchon_opencl_lib_amd.layers import Linear

_glob = None


def glob():
    global _glob
    if _glob is None:
        _glob = NnClGlob("cuda:0")
    return _glob


def listed():
    return [
        # the 256^3 product: the smallest ordinary call, where latency and launches count
        {"name": "matmul_256", "kind": "matmul", "m": 256, "k": 256, "n": 256},
        # no dimension a multiple of any tile: dynamic sizes
        {"name": "matmul_ragged", "kind": "matmul", "m": 1000, "k": 777, "n": 3000},
        # the headline: 4096^3 forward with both gradients (the largest case)
        {"name": "square_train", "kind": "square_train", "m": 4096, "k": 4096, "n": 4096},
        # 4 sequences x 8 heads of 128 tokens, head width 64
        {"name": "attention", "kind": "attention", "heads": 32, "seq": 128, "dim": 64},
        # a vision-like sequence of odd length, more heads
        {"name": "attention_ragged", "kind": "attention", "heads": 48, "seq": 197, "dim": 72},
        # the encoder/decoder's output layer: Linear(500 -> 6565) on [8, 1500, 500]
        {"name": "linear_train", "kind": "linear_train", "batch": 8, "rows": 1500, "fin": 500,
         "fout": 6565},
        # a single token through a wide layer: bound by reading the weight
        {"name": "decode_row", "kind": "decode", "rows": 1, "fin": 4096, "fout": 11008,
         "stored_nk": False},
        # a small serving batch through the layer's [out, in] weight
        {"name": "decode_batch", "kind": "decode", "rows": 24, "fin": 2048, "fout": 4096,
         "stored_nk": True},
        # one recurrent step of 64 sequences, input 512, hidden 1024
        {"name": "lstm_step", "kind": "lstm_step", "batch": 64, "fin": 512, "hidden": 1024},
        # the same LSTM over 100 steps: every GEMM stage of forward and backward
        {"name": "lstm_train", "kind": "lstm_train", "batch": 64, "seq": 100, "fin": 512,
         "hidden": 1024},
        # splitting heads: [batch, seq, heads, dim] -> [batch, heads, dim, seq]
        {"name": "permute_heads", "kind": "permute", "shape": "32x500x16x64", "axes": "0231"},
        # reducing the last axis (row sums of a score matrix)
        {"name": "sum_rows", "kind": "sum", "shape": "64x1000x513", "axis": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size over [lo, hi], log-uniform; every second one rounded to a multiple of 32 (the
    widths of layers), the others as they fall, odd ones among them."""
    v = _log_int(rng, lo, hi)
    if rng.random() < 0.5 and v >= 32:
        v = v // 32 * 32
    return v


def draw(rng):
    kind = rng.choice(["matmul", "square_train", "attention", "linear_train", "decode",
                       "lstm_step", "lstm_train", "permute", "sum"])
    if kind == "matmul":
        return {"kind": kind, "m": _size(rng, 16, 3000), "k": _size(rng, 16, 3000),
                "n": _size(rng, 16, 3000)}
    if kind == "square_train":
        return {"kind": kind, "m": _size(rng, 500, 4096), "k": _size(rng, 500, 4096),
                "n": _size(rng, 500, 4096)}
    if kind == "attention":
        return {"kind": kind, "heads": _log_int(rng, 4, 96), "seq": _size(rng, 20, 600),
                "dim": rng.choice([32, 40, 64, 72, 80, 96, 128])}
    if kind == "linear_train":
        return {"kind": kind, "batch": _log_int(rng, 1, 16), "rows": _size(rng, 50, 1500),
                "fin": _size(rng, 64, 1500), "fout": _size(rng, 64, 6565)}
    if kind == "decode":
        return {"kind": kind, "rows": _log_int(rng, 1, 64), "fin": _size(rng, 256, 8192),
                "fout": _size(rng, 256, 11008), "stored_nk": rng.random() < 0.5}
    if kind == "lstm_step":
        return {"kind": kind, "batch": _log_int(rng, 1, 128), "fin": _size(rng, 32, 1024),
                "hidden": _size(rng, 64, 1024)}
    if kind == "lstm_train":
        return {"kind": kind, "batch": _log_int(rng, 4, 64), "seq": _log_int(rng, 10, 100),
                "fin": _size(rng, 32, 1024), "hidden": _size(rng, 64, 1024)}
    if kind == "permute":
        dims, axes = rng.choice([
            ((_log_int(rng, 200, 6000), _log_int(rng, 200, 6000)), "10"),
            ((_log_int(rng, 2, 64), _log_int(rng, 30, 600), _log_int(rng, 30, 600)), "021"),
            ((_log_int(rng, 2, 64), _log_int(rng, 30, 600), _log_int(rng, 30, 600)),
             rng.choice(["102", "120", "201", "210"])),
            ((_log_int(rng, 2, 32), _log_int(rng, 20, 512), _log_int(rng, 2, 16),
              rng.choice([32, 50, 64, 80])), rng.choice(["0213", "0231", "2013", "0312"])),
        ])
        return {"kind": kind, "shape": "x".join(map(str, dims)), "axes": axes}
    dims = (_log_int(rng, 1, 64), _log_int(rng, 20, 1500), _log_int(rng, 20, 1500))
    while dims[0] * dims[1] * dims[2] > 40_000_000:
        dims = (max(1, dims[0] // 2),) + dims[1:]
    return {"kind": "sum", "shape": "x".join(map(str, dims)), "axis": rng.randrange(3)}


def _dims(case):
    return [int(v) for v in case["shape"].split("x")]


def _axes(case):
    return [int(v) for v in case["axes"]]


class _Values:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda:0").manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda:0") * std

    def uniform(self, *shape, bound=1.0):
        return (torch.rand(shape, generator=self.g, device="cuda:0") * 2 - 1) * bound


def _tensors(case, seed):
    """The inputs of a case, by name."""
    v = _Values(seed)
    kind = case["kind"]
    if kind == "matmul":
        return {"a": v.uniform(1, case["m"], case["k"]), "b": v.uniform(1, case["k"], case["n"])}
    if kind == "square_train":
        s = 1.0 / math.sqrt(case["k"])
        return {"a": v.normal(1, case["m"], case["k"], std=s),
                "b": v.normal(1, case["k"], case["n"], std=s),
                "dc": v.normal(1, case["m"], case["n"], std=s)}
    if kind == "attention":
        h, s, d = case["heads"], case["seq"], case["dim"]
        return {"q": v.normal(h, s, d), "kt": v.normal(h, d, s),
                "p": torch.softmax(v.normal(h, s, s), dim=-1), "v": v.normal(h, s, d),
                "ds": v.normal(h, s, s, std=0.1), "do": v.normal(h, s, d, std=0.1)}
    if kind == "linear_train":
        b, r, i, o = case["batch"], case["rows"], case["fin"], case["fout"]
        bound = 1.0 / math.sqrt(i)
        return {"x": v.normal(b, r, i), "w": v.uniform(1, i, o, bound=bound),
                "bias": v.uniform(o, bound=bound), "gy": v.normal(b, r, o, std=0.01)}
    if kind == "decode":
        i, o = case["fin"], case["fout"]
        shape = (o, i) if case["stored_nk"] else (i, o)
        return {"x": v.normal(case["rows"], i), "w": v.uniform(*shape, bound=1.0 / math.sqrt(i))}
    if kind == "lstm_step":
        b, f, h = case["batch"], case["fin"], case["hidden"]
        bound = 1.0 / math.sqrt(h)
        return {"x": v.normal(b, 2, f), "w": v.uniform(f, 4 * h, bound=bound),
                "u": v.uniform(h, 4 * h, bound=bound), "bias": v.uniform(4 * h, bound=bound),
                "hprev": v.uniform(b, h), "hout": v.uniform(b, 2, h)}
    if kind == "lstm_train":
        b, s, f, h = case["batch"], case["seq"], case["fin"], case["hidden"]
        bound = 1.0 / math.sqrt(h)
        return {"x": v.normal(b, s, f), "w": v.uniform(f, 4 * h, bound=bound),
                "bias": v.uniform(4 * h, bound=bound), "hout": v.uniform(b, s, h),
                "g": v.normal(b * s, 4 * h, std=0.01)}
    if kind == "permute":
        return {"x": v.normal(*_dims(case))}
    if kind == "sum":
        return {"x": v.uniform(*_dims(case)) + 0.5}
    raise ValueError(kind)


def prepare(case, seed):
    state = dict(_tensors(case, seed), case=case)
    kind = case["kind"]
    if kind == "linear_train":
        for name in ("x", "w", "bias"):
            state[name].requires_grad_(True)
    elif kind == "decode" and case["stored_nk"]:
        state["layer"] = Linear(case["fin"], case["fout"], nnclglob=glob(), weight=state["w"])
    elif kind == "lstm_step":
        state["workspace"] = torch.empty(2, case["batch"], 4 * case["hidden"], device="cuda:0")
    elif kind == "lstm_train":
        state["dw"] = torch.zeros_like(state["w"])
        state["du"] = torch.zeros(case["hidden"], 4 * case["hidden"], device="cuda:0")
        state["db"] = torch.zeros_like(state["bias"])
    return state


def run(state):
    case, g = state["case"], glob()
    kind = case["kind"]
    if kind == "matmul":
        return g.Bmm(state["a"], state["b"])
    if kind == "square_train":
        c = g.Bmm(state["a"], state["b"])
        da, db = g.bmm_backward(state["dc"], state["a"], state["b"])
        return c, da, db
    if kind == "attention":
        s = g.Bmm(state["q"], state["kt"])
        o = g.Bmm(state["p"], state["v"])
        dp, dv = g.bmm_backward(state["do"], state["p"], state["v"])
        dq, dkt = g.bmm_backward(state["ds"], state["q"], state["kt"])
        return s, o, dp, dv, dq, dkt
    if kind == "linear_train":
        y = linear(state["x"], state["w"], state["bias"])
        return (y,) + torch.autograd.grad(y, (state["x"], state["w"], state["bias"]), state["gy"])
    if kind == "decode":
        return state["layer"](state["x"]) if "layer" in state else g.gemm(state["x"], state["w"])
    if kind == "lstm_step":
        # the second step of a chunk: h_{t-1} is the first step's row of hout
        return g.LstmHidGates(state["x"], state["w"], state["u"], state["bias"], state["hprev"],
                              state["hout"], state["workspace"], 1)[1]
    if kind == "lstm_train":
        xw = g.LstmGemmXW(state["x"], state["w"], state["bias"])
        for name in ("dw", "du", "db"):  # the training loop's zero_grad()
            state[name].zero_()
        dx = g.LstmGemmGradX(state["g"], state["w"], state["x"].shape)
        g.LstmGemmGradWeights(state["x"], state["hout"], state["g"], state["dw"], state["du"],
                              state["db"])
        return xw, dx, state["dw"], state["du"], state["db"]
    if kind == "permute":
        return g.Permute(state["x"], _axes(case))
    if kind == "sum":
        return g.Sum(state["x"], case["axis"])
    raise ValueError(kind)


def _products(case):
    """(flops, floats read, floats written) of one pass."""
    kind = case["kind"]
    if kind in ("matmul", "square_train"):
        m, k, n = case["m"], case["k"], case["n"]
        one = 2 * m * k * n
        if kind == "matmul":
            return one, m * k + k * n, m * n
        return 3 * one, m * k + k * n + m * n, m * n + m * k + k * n
    if kind == "attention":
        h, s, d = case["heads"], case["seq"], case["dim"]
        return 6 * 2 * h * s * s * d, h * (4 * s * d + 2 * s * s), h * (4 * s * d + 2 * s * s)
    if kind == "linear_train":
        t, i, o = case["batch"] * case["rows"], case["fin"], case["fout"]
        return 6 * t * i * o, t * i + i * o + o + t * o, t * o + t * i + i * o + o
    if kind == "decode":
        r, i, o = case["rows"], case["fin"], case["fout"]
        return 2 * r * i * o, r * i + i * o, r * o
    if kind == "lstm_step":
        b, f, h = case["batch"], case["fin"], case["hidden"]
        return 2 * b * (f + h) * 4 * h, b * (f + h) + (f + h + 1) * 4 * h, b * 4 * h
    if kind == "lstm_train":
        t, f, h = case["batch"] * case["seq"], case["fin"], case["hidden"]
        return (2 * t * 4 * h * (3 * f + h), t * (f + h + 4 * h) + (f + 1) * 4 * h,
                t * (4 * h + f) + (f + h + 1) * 4 * h)
    n = int(np.prod(_dims(case)))
    if kind == "permute":
        return 0, n, n
    return n, n, n // _dims(case)[case["axis"]]


def work(case):
    flops, read, written = _products(case)
    return {"bytes": 4 * (read + written), "flops": flops}


def _longest_sum(case):
    kind = case["kind"]
    if kind == "matmul":
        return case["k"]
    if kind == "square_train":
        return max(case["m"], case["k"], case["n"])
    if kind == "attention":
        return max(case["seq"], case["dim"])
    if kind == "linear_train":
        return max(case["batch"] * case["rows"], case["fin"], case["fout"])
    if kind == "decode":
        return case["fin"]
    if kind == "lstm_step":
        return case["fin"] + case["hidden"]
    if kind == "lstm_train":
        return max(case["batch"] * case["seq"], 4 * case["hidden"], case["fin"])
    return _dims(case)[case["axis"]]


def tolerance(case):
    """fp32 sums of random values against 64 bits: 1.1e-7 to 1.5e-7 over short sums, then
    1.8e-8 sqrt(k) for a k-long one (1.1e-6 at k = 4096); four times that. The largest single
    difference of some 10^7 outputs is six to eight standard deviations."""
    if case["kind"] == "permute":
        return "exact"
    rel = 6e-7 + 7.2e-8 * math.sqrt(_longest_sum(case))
    return {"rel": rel, "max": 10 * rel}


def exact(case, seed):
    t = {name: x.double() for name, x in _tensors(case, seed).items()}
    kind = case["kind"]
    if kind == "matmul":
        return t["a"] @ t["b"]
    if kind == "square_train":
        return (t["a"] @ t["b"], t["dc"] @ t["b"].transpose(1, 2).contiguous(),
                t["a"].transpose(1, 2).contiguous() @ t["dc"])
    if kind == "attention":
        tr = lambda x: x.transpose(1, 2).contiguous()  # noqa: E731
        return (t["q"] @ t["kt"], t["p"] @ t["v"], t["do"] @ tr(t["v"]), tr(t["p"]) @ t["do"],
                t["ds"] @ tr(t["kt"]), tr(t["q"]) @ t["ds"])
    if kind == "linear_train":
        i, o = case["fin"], case["fout"]
        x, w, gy = t["x"].reshape(-1, i), t["w"].reshape(i, o), t["gy"].reshape(-1, o)
        lead = (case["batch"], case["rows"])
        return ((x @ w + t["bias"]).reshape(*lead, o), (gy @ w.t()).reshape(*lead, i),
                (x.t() @ gy).reshape(1, i, o), gy.sum(0))
    if kind == "decode":
        return t["x"] @ (t["w"].t() if case["stored_nk"] else t["w"])
    if kind == "lstm_step":
        return t["bias"] + t["x"][:, 1] @ t["w"] + t["hout"][:, 0] @ t["u"]
    if kind == "lstm_train":
        f, h = case["fin"], case["hidden"]
        x, gg = t["x"].reshape(-1, f), t["g"]
        before = torch.zeros_like(t["hout"])
        before[:, 1:] = t["hout"][:, :-1]
        return (x @ t["w"] + t["bias"], (gg @ t["w"].t()).reshape(t["x"].shape), x.t() @ gg,
                before.reshape(-1, h).t() @ gg, gg.sum(0))
    if kind == "permute":
        return t["x"].permute(_axes(case)).contiguous()
    return t["x"].sum(case["axis"])
