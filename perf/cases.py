"""What a program built on deepfuse_amd has it do: fp8 Linear layers and what stands around them.

A case is a dict of plain values; its "kind" says which part of the library it runs:

  model      the Linears of one or more blocks: quantize the activations just in time, forward, and with
             "backward" also the gradients' quantize, dX, dW and db; "weights" says whether the program keeps
             fp8 codes ("codes", inference) or quantizes its master weights on each pass ("master", training);
             with "graph" the pass is captured once and replayed, as a launch-bound program does
  backward   one Linear's backward on its own, from the upstream gradient to dX, dW and db
  mlp        fc1 -> fc2 of a block, the activations at delayed scaling, fc1's output scale from its GEMM
  convert    a flat tensor to fp8 and back: absmax, scale, quantize, dequantize
  layernorm  LayerNorm whose output leaves as fp8 codes (row and transposed)
  optimizer  gradient clipping, Adam and the updated weights' fp8 codes

The sizes are those of GPT-2 small and GPT-2 XL Linears, as bench.py and the tests run them, and odd ones.
"""
import ctypes
import math

import numpy as np
import torch

import deepfuse_amd as df
from deepfuse_amd import DType, Fmt

SMALL = "768x2304,768x768,768x3072,3072x768"  # in x out of one GPT-2 small block's Linears
XL = "1600x4800,1600x1600,1600x6400,6400x1600"  # and of a GPT-2 XL block's

TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
CODE = {"f32": int(DType.FLOAT32), "bf16": int(DType.BFLOAT16), "f16": int(DType.HALF)}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
FMT = {"e4m3": Fmt.E4M3, "e5m2": Fmt.E5M2}
FMAX = {"e4m3": 448.0, "e5m2": 57344.0}
F8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
E4, E5 = int(Fmt.E4M3), int(Fmt.E5M2)


def model(name, tokens, linears, dtype="bf16", layers=1, weights="master", backward=False, graph=False):
    return {"name": name, "kind": "model", "tokens": tokens, "linears": linears, "dtype": dtype, "layers": layers,
            "weights": weights, "backward": backward, "graph": graph}


def listed():
    return [
        # one layer called for a handful of tokens in fp32: the smallest call, all latency
        model("linear_fp32_64", 64, "768x3072", dtype="f32", weights="codes"),
        # generation: a few sequences through the Linears of six XL blocks, bound by reading the weights once
        model("decode_xl_8", 8, XL, layers=6, weights="codes", graph=True),
        # a training step on a small batch of a small model, captured because it is launch-bound
        model("step_small_512", 512, SMALL, backward=True, graph=True),
        # a small model's forward over a full batch (8 x 1024 tokens), weights quantized on each pass
        model("forward_small_8192", 8192, SMALL),
        # one large Linear's forward, weights kept as codes
        model("forward_xl_fc", 16384, "1600x6400", weights="codes"),
        # one large Linear's backward
        {"name": "backward_xl_qkv", "kind": "backward", "tokens": 16384, "k": 1600, "n": 4800, "dtype": "bf16"},
        # the Linears of a large model's block, forward and backward, weights quantized on each pass: the headline step
        model("step_xl_16384", 16384, XL, backward=True),
        # a layer of odd sizes in half precision, forward and backward
        model("step_ragged_f16", 1000, "771x1037", dtype="f16", backward=True),
        # a tensor converted to fp8 and back, outliers and non-finite values among it
        {"name": "convert_f32", "kind": "convert", "n": 134217728, "src": "f32", "fmt": "e4m3"},
        # the producer of a large model's qkv and fc inputs
        {"name": "layernorm_xl", "kind": "layernorm", "rows": 16384, "cols": 1600, "dtype": "bf16"},
        # the consumer of a large model's gradients: two blocks' weights
        {"name": "optimizer_xl_2", "kind": "optimizer", "layers": 2, "linears": XL},
        # a block's fc1 -> fc2 over an ordinary batch at delayed scaling
        {"name": "mlp_xl_4096", "kind": "mlp", "tokens": 4096, "d": 1600, "h": 6400},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo=64, hi=6400):
    """A layer width: any number, or, as most models have them, a multiple of 64."""
    w = _log(rng, lo, hi)
    return w if rng.random() < 0.4 else max(64, (w + 32) // 64 * 64)


MOST = {"bytes": 1.2e9, "flops": 2.5e12}  # a drawn case stays below the largest listed ones


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if all(w[k] <= MOST[k] for k in MOST):
            return c


def _draw(rng):
    kind = rng.choice(["linear", "linear", "decode", "step", "step", "backward", "mlp", "convert", "layernorm",
                       "optimizer"])
    if kind in ("linear", "step"):
        train = kind == "step"
        count = rng.choice([1, 1, 2, 4])
        lin = ",".join("%dx%d" % (_width(rng), _width(rng)) for _ in range(count))
        tokens = _log(rng, 16, 16384)
        c = model("", tokens, lin, dtype=rng.choice(["bf16", "bf16", "f16", "f32"]),
                  weights="master" if train else rng.choice(["codes", "master"]), backward=train,
                  graph=tokens <= 2048 and rng.random() < 0.6)
    elif kind == "decode":
        lin = ",".join("%dx%d" % (_width(rng, 256), _width(rng, 256)) for _ in range(rng.choice([2, 4])))
        c = model("", _log(rng, 1, 64), lin, layers=rng.choice([1, 2, 4, 6]), weights="codes", graph=True)
    elif kind == "backward":
        return {"kind": kind, "tokens": _log(rng, 16, 16384), "k": _width(rng), "n": _width(rng, 64, 4800),
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"])}
    elif kind == "mlp":
        return {"kind": kind, "tokens": _log(rng, 64, 8192), "d": _width(rng, 256, 1600), "h": _width(rng, 1024, 6400)}
    elif kind == "convert":
        return {"kind": kind, "n": _log(rng, 1000, 134217728), "src": rng.choice(["f32", "bf16"]),
                "fmt": rng.choice(["e4m3", "e5m2"])}
    elif kind == "layernorm":
        return {"kind": kind, "rows": _log(rng, 64, 16384), "cols": _width(rng, 128, 6400),
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"])}
    else:
        lin = ",".join("%dx%d" % (_width(rng), _width(rng)) for _ in range(rng.choice([1, 2, 4])))
        return {"kind": kind, "layers": rng.choice([1, 2, 3]), "linears": lin}
    del c["name"]
    return c


# ---- sizes, inputs ---------------------------------------------------------------------------------------------------

def _linears(case):
    return [tuple(int(v) for v in p.split("x")) for p in case["linears"].split(",")]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, std, dtype):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _model_inputs(case, seed):
    """Per Linear (layer by layer): activations X [M, K], weights W [N, K], bias [N] and, with "backward", the
    upstream gradient dY [M, N]."""
    g, dt, M = _gen(seed), TORCH[case["dtype"]], case["tokens"]
    out = []
    for _ in range(case["layers"]):
        for K, N in _linears(case):
            out.append({"K": K, "N": N, "x": _normal(g, (M, K), 1.0, dt), "w": _normal(g, (N, K), 0.02, dt),
                        "b": _normal(g, (N,), 0.02, dt),
                        "dy": _normal(g, (M, N), 1e-3, dt) if case["backward"] else None})
    return out


def _backward_inputs(case, seed):
    g, dt = _gen(seed), TORCH[case["dtype"]]
    M, K, N = case["tokens"], case["k"], case["n"]
    return {"x": _normal(g, (M, K), 1.0, dt), "w": _normal(g, (N, K), 0.02, dt), "dy": _normal(g, (M, N), 1e-3, dt)}


def _mlp_inputs(case, seed):
    g, bf, M, d, h = _gen(seed), torch.bfloat16, case["tokens"], case["d"], case["h"]
    return {"x": _normal(g, (M, d), 1.0, bf), "w1": _normal(g, (h, d), 0.02, bf), "b1": _normal(g, (h,), 0.02, bf),
            "w2": _normal(g, (d, h), 0.02, bf), "b2": _normal(g, (d,), 0.02, bf)}


def _convert_input(case, seed):
    """N(0, 1), 0.1% of the values a thousand times larger, and the non-finite and tiny values that turn up."""
    g, n = _gen(seed), case["n"]
    x = torch.randn(n, generator=g, device="cuda")
    at = torch.randint(0, n, (max(1, n // 1000),), generator=g, device="cuda")
    x[at] *= 1000.0
    special = torch.tensor([math.inf, -math.inf, math.nan, 1e-40, -1e-40, 0.0, -0.0], device="cuda")
    x[torch.randperm(min(n, 100000), generator=g, device="cuda")[:len(special)]] = special
    return x.to(TORCH[case["src"]])


def _layernorm_inputs(case, seed):
    g, dt = _gen(seed), TORCH[case["dtype"]]
    return {"x": _normal(g, (case["rows"], case["cols"]), 2.0, torch.float32).add_(0.25).to(dt),
            "gamma": (_normal(g, (case["cols"],), 0.1, torch.float32) + 1.0).to(dt),
            "beta": _normal(g, (case["cols"],), 0.1, dt)}


def _optimizer_inputs(case, seed):
    """Weights and biases of every Linear, their gradients and Adam's moments after some steps."""
    g = _gen(seed)
    shapes = [s for _ in range(case["layers"]) for K, N in _linears(case) for s in ((N, K), (N,))]
    f32 = torch.float32
    return {"p": [_normal(g, s, 0.02, f32) for s in shapes], "g": [_normal(g, s, 1e-3, f32) for s in shapes],
            "m": [_normal(g, s, 1e-4, f32) for s in shapes],
            "v": [_normal(g, s, 1e-3, f32).square_() for s in shapes]}


CLIP, LR, EPS, STEP = 1.0, 1e-3, 1e-8, 10


# ---- the programs ----------------------------------------------------------------------------------------------------

def _u8(rows, cols):
    return torch.empty((rows, cols), dtype=torch.uint8, device="cuda")


def _ptr(t):
    return None if t is None else t.data_ptr()


class Model:
    """Linears with their buffers and workspaces allocated once, driven through the C ABI."""

    def __init__(self, case, inputs):
        self.M, self.dt, self.backward = case["tokens"], case["dtype"], case["backward"]
        self.master = case["weights"] == "master"
        L, M, r16, train = df.lib(), self.M, df.round16, self.backward
        dt = TORCH[self.dt]
        self.dw_dt = torch.float16 if self.dt == "f16" else torch.float32
        self.lin, jit, gemm = [], 16, 16
        for a in inputs:
            K, N = a["K"], a["N"]
            s = dict(a, xq=_u8(M, r16(K)), wq=_u8(N, r16(K)), wt=_u8(K, r16(N)) if train else None,
                     xt=_u8(K, r16(M)) if train else None, y=torch.empty((M, N), dtype=dt, device="cuda"),
                     sc=torch.zeros(8, device="cuda"))
            jit = max(jit, *(L.df_quantize_2d_jit_workspace_bytes(r, c, 1) for r, c in ((M, K), (N, K), (M, N))))
            gemm = max(gemm, L.df_fp8_gemm_workspace_bytes(M, N, K))
            if train:
                s.update(dyq=_u8(M, r16(N)), dyt=_u8(N, r16(M)), dx=torch.empty((M, K), dtype=dt, device="cuda"),
                         dw=torch.empty((N, K), dtype=self.dw_dt, device="cuda"), db=torch.empty(N, device="cuda"))
                gemm = max(gemm, L.df_fp8_gemm_bwd_workspace_bytes(M, N, K))
            self.lin.append(s)
        self.jit, self.gemm = _u8(1, jit), _u8(1, gemm)
        # weights of one block in one call (fp32 and bf16), as after an optimizer step
        self.sw = torch.empty(len(self.lin), device="cuda")
        self.batched = self.dt != "f16" and len(self.lin) > 1
        if self.batched:
            n = len(self.lin)
            ptrs = lambda k: (ctypes.c_void_p * n)(*[_ptr(s[k]) for s in self.lin])  # noqa: E731
            ints = lambda v: (ctypes.c_int * n)(*v)  # noqa: E731
            self.bws = _u8(1, L.df_quantize_2d_batch_workspace_bytes())
            self.bargs = (CODE[self.dt], n, ptrs("w"), ints([s["N"] for s in self.lin]),
                          ints([s["K"] for s in self.lin]), E4, None, _ptr(self.sw), ptrs("wq"),
                          ints([r16(s["K"]) for s in self.lin]), ptrs("wt") if train else None,
                          ints([r16(s["N"]) for s in self.lin]) if train else None, _ptr(self.bws), self.bws.numel())
        if not self.master:
            self.weights()
        self.graph = None
        if case["graph"]:
            self.step()  # warm-up
            torch.cuda.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                self.step()

    def quantize(self, x, rows, cols, fmt, sc, q, qt, colsum=None):
        df.call("df_quantize_2d_jit", CODE[self.dt], _ptr(x), rows, cols, fmt, None, sc, _ptr(q),
                q.shape[1] if q is not None else 0, _ptr(qt), qt.shape[1] if qt is not None else 0, _ptr(colsum),
                _ptr(self.jit), self.jit.numel(), torch.cuda.current_stream().cuda_stream)

    def weights(self):
        if self.batched:
            df.call("df_quantize_2d_batch", *self.bargs, torch.cuda.current_stream().cuda_stream)
        else:
            for i, s in enumerate(self.lin):
                self.quantize(s["w"], s["N"], s["K"], E4, _ptr(self.sw) + 4 * i, s["wq"], s["wt"])

    def step(self):
        M, dt, st = self.M, CODE[self.dt], torch.cuda.current_stream().cuda_stream
        if self.master:
            self.weights()
        for i, s in enumerate(self.lin):
            K, N, sx = s["K"], s["N"], _ptr(s["sc"])
            self.quantize(s["x"], M, K, E4, sx, s["xq"], s["xt"])
            df.call("df_fp8_gemm_fwd", _ptr(s["xq"]), s["xq"].shape[1], _ptr(s["wq"]), s["wq"].shape[1], M, N, K, sx,
                    _ptr(self.sw) + 4 * i, dt, _ptr(s["b"]), dt, _ptr(s["y"]), N, _ptr(self.gemm), self.gemm.numel(),
                    st)
        if self.backward:
            dw_dt = CODE["f16"] if self.dt == "f16" else CODE["f32"]
            for i in reversed(range(len(self.lin))):
                s = self.lin[i]
                K, N, sx, sdy = s["K"], s["N"], _ptr(s["sc"]), _ptr(s["sc"]) + 4
                self.quantize(s["dy"], M, N, E5, sdy, s["dyq"], s["dyt"], s["db"])
                df.call("df_fp8_gemm_bwd", _ptr(s["dyq"]), s["dyq"].shape[1], _ptr(s["wt"]), s["wt"].shape[1],
                        _ptr(s["dyt"]), s["dyt"].shape[1], _ptr(s["xt"]), s["xt"].shape[1], M, N, K, sdy,
                        _ptr(self.sw) + 4 * i, sx, dt, _ptr(s["dx"]), K, dw_dt, _ptr(s["dw"]), K, _ptr(self.gemm),
                        self.gemm.numel(), st)

    def run(self):
        if self.graph is not None:
            self.graph.replay()
        else:
            self.step()
        return {k: [s[k] for s in self.lin] for k in (("y", "dx", "dw", "db") if self.backward else ("y",))}


class Backward:
    """One Linear's backward; its forward left the codes of X and W."""

    def __init__(self, case, a):
        M, K, N, dt = case["tokens"], case["k"], case["n"], case["dtype"]
        L, r16 = df.lib(), df.round16
        self.shape, self.dt, self.dy = (M, K, N), CODE[dt], a["dy"]
        _, self.sx, _, self.xt = df.quantize_2d_jit(a["x"], Fmt.E4M3, want_q=False, want_qt=True)
        _, self.sw, _, self.wt = df.quantize_2d_jit(a["w"], Fmt.E4M3, want_q=False, want_qt=True)
        self.dyq, self.dyt, self.sdy = _u8(M, r16(N)), _u8(N, r16(M)), torch.empty(1, device="cuda")
        self.dw_dt = "f16" if dt == "f16" else "f32"
        self.dx = torch.empty((M, K), dtype=TORCH[dt], device="cuda")
        self.dw = torch.empty((N, K), dtype=TORCH[self.dw_dt], device="cuda")
        self.db = torch.empty(N, device="cuda")
        self.jit = _u8(1, L.df_quantize_2d_jit_workspace_bytes(M, N, 1))
        self.gemm = _u8(1, max(16, L.df_fp8_gemm_bwd_workspace_bytes(M, N, K)))

    def run(self):
        (M, K, N), st = self.shape, torch.cuda.current_stream().cuda_stream
        df.call("df_quantize_2d_jit", self.dt, _ptr(self.dy), M, N, E5, None, _ptr(self.sdy), _ptr(self.dyq),
                self.dyq.shape[1], _ptr(self.dyt), self.dyt.shape[1], _ptr(self.db), _ptr(self.jit),
                self.jit.numel(), st)
        df.call("df_fp8_gemm_bwd", _ptr(self.dyq), self.dyq.shape[1], _ptr(self.wt), self.wt.shape[1],
                _ptr(self.dyt), self.dyt.shape[1], _ptr(self.xt), self.xt.shape[1], M, N, K, _ptr(self.sdy),
                _ptr(self.sw), _ptr(self.sx), self.dt, _ptr(self.dx), K, CODE[self.dw_dt], _ptr(self.dw), K,
                _ptr(self.gemm), self.gemm.numel(), st)
        return {"dx": self.dx, "dw": self.dw, "db": self.db}


class Mlp:
    """fc1 -> fc2: X at delayed scaling, fc1's output quantized at the scale its GEMM gave."""

    def __init__(self, case, a):
        self.a, self.d, self.h = a, case["d"], case["h"]
        _, (self.s1, self.s2), (self.w1, self.w2), _ = self._weights(a)
        amax, _ = df.absmax_scale(a["x"], Fmt.E4M3)
        self.hist = df.DelayedScale(Fmt.E4M3, 16, a["x"].device, seed_amax=amax)

    @staticmethod
    def _weights(a):
        am, sc, q, qt = df.quantize_2d_batch([a["w1"], a["w2"]], Fmt.E4M3, want_qt=False)
        return am, (sc[:1], sc[1:]), q, qt

    def run(self):
        a, E = self.a, Fmt.E4M3
        scale = self.hist.scale.clone()
        xq, _ = self.hist.quantize_2d(a["x"])
        y1, _, sy = df.gemm_fwd_absmax(xq, self.w1, self.d, scale, self.s1, bias=a["b1"], next_fmt=E)
        yq, _ = df.quantize_2d(y1, sy, E)
        y2 = df.gemm_nt(yq, E, self.w2, E, self.h, sy, self.s2, bias=a["b2"], out_dtype=torch.bfloat16)
        return {"y1": y1, "y2": y2}


class Convert:
    def __init__(self, case, x):
        self.x, self.fmt = x, FMT[case["fmt"]]

    def run(self):
        am, sc = df.absmax_scale(self.x, self.fmt)
        q = df.quantize(self.x, sc, self.fmt)
        return {"absmax": am, "scale": sc, "codes": q, "back": df.dequantize(q, sc, self.fmt, self.x.dtype)}


class LayerNorm:
    def __init__(self, case, a):
        self.a = a

    def run(self):
        _, q, qt, sc = df.layernorm(self.a["x"], self.a["gamma"], self.a["beta"], fmt=Fmt.E4M3, want_y=False,
                                    want_qt=True)
        return {"q": q[:, :self.a["x"].shape[1]], "qt": qt[:, :self.a["x"].shape[0]], "scale": sc}


class Optimizer:
    def __init__(self, case, a):
        self.a, self.t = a, STEP
        self.absmax = torch.empty(len(a["p"]), device="cuda")
        self.w = [i for i, p in enumerate(a["p"]) if p.dim() == 2]

    def run(self):
        a = self.a
        norm = df.grad_norm(a["g"])
        df.adam_update(a["p"], a["g"], a["m"], a["v"], self.t, lr=LR, eps=EPS, clip_norm=norm, max_norm=CLIP,
                       absmax=self.absmax)
        self.t += 1
        _, sc, q, qt = df.quantize_2d_batch([a["p"][i] for i in self.w], Fmt.E4M3, absmax=self.absmax[::2].contiguous())
        # the first and last weight whole, with their moments and codes: every tensor takes the same path
        ends = (self.w[0], self.w[-1])
        return {"norm": norm, "absmax": self.absmax, "scale": sc, "p": [a["p"][i] for i in ends],
                "m": [a["m"][i] for i in ends], "v": [a["v"][i] for i in ends], "b": a["p"][-1],
                "q": [q[0], q[-1]], "qt": [qt[0], qt[-1]]}


KINDS = {"model": (Model, _model_inputs), "backward": (Backward, _backward_inputs), "mlp": (Mlp, _mlp_inputs),
         "convert": (Convert, _convert_input), "layernorm": (LayerNorm, _layernorm_inputs),
         "optimizer": (Optimizer, _optimizer_inputs)}


def prepare(case, seed):
    program, inputs = KINDS[case["kind"]]
    return program(case, inputs(case, seed))


def run(state):
    return state.run()


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "model":
        M, e, b, f = case["tokens"], SIZE[case["dtype"]], 0, 0
        for K, N in _linears(case) * case["layers"]:
            w = N * K * (e if case["weights"] == "master" else 1)
            b += e * M * (K + N) + w + e * N  # X, Y, W, bias
            f += 2 * M * N * K
            if case["backward"]:
                b += e * M * (K + N) + N * K * (2 if case["dtype"] == "f16" else 4) + 4 * N  # dY, dX, dW, db
                f += 4 * M * N * K
        return {"bytes": b, "flops": f}
    if kind == "backward":
        M, K, N, e = case["tokens"], case["k"], case["n"], SIZE[case["dtype"]]
        return {"bytes": e * M * (N + K) + N * K + M * K + N * K * (2 if case["dtype"] == "f16" else 4) + 4 * N,
                "flops": 4 * M * N * K}
    if kind == "mlp":
        M, d, h = case["tokens"], case["d"], case["h"]
        return {"bytes": 2 * M * (2 * d + h) + 2 * d * h + 2 * (d + h), "flops": 4 * M * d * h}
    if kind == "convert":
        return {"bytes": case["n"] * (2 * SIZE[case["src"]] + 1), "flops": 0}
    if kind == "layernorm":
        n = case["rows"] * case["cols"]
        return {"bytes": n * (SIZE[case["dtype"]] + 2), "flops": 8 * n}
    n = sum(K * N for K, N in _linears(case)) * case["layers"]
    b = sum(N for K, N in _linears(case)) * case["layers"]
    return {"bytes": 28 * (n + b) + 2 * n, "flops": 16 * (n + b)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("convert", "layernorm"):
        # codes, scales and the values they stand for are fixed bit for bit by the conversion's definition
        return "exact"
    if kind == "optimizer":
        # 32-bit arithmetic in a stated order; the norm is a sum in 64 bits, rounded once
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    # The matrix units sum fp8 products in 32 bits with a short alignment: another order of a sum moves an fp32 result by
    # 1.6e-5 (2-norm; 1.5e-4 at most). Rounded to 16 bits, some results land one unit in the last place away: 2.4e-4
    # and 7.8e-3 in bf16, 8.5e-5 and 9.8e-4 in f16. Four times these.
    if kind == "mlp":
        # fc1's changed roundings change some of fc2's input codes, a unit of three bits each: 1.7e-3 and 1.8e-2
        return {"rel": 7e-3, "max": 8e-2}
    return {"f32": {"rel": 6.4e-5, "max": 6e-4}, "f16": {"rel": 3.4e-4, "max": 4e-3},
            "bf16": {"rel": 1e-3, "max": 3.2e-2}}[case["dtype"]]


# ---- the same in 64 bits, in plain torch -----------------------------------------------------------------------------

def _scale(x, fmt):
    """absmax over the finite values, and absmax / largest code, both binary32 by definition."""
    a = x.float().abs()
    am = torch.where(torch.isfinite(a), a, torch.zeros_like(a)).amax()
    s = am / torch.full_like(am, FMAX[fmt])  # by a tensor: torch divides by a number as a product, which rounds twice
    return am, torch.where(s > 0, s, torch.ones_like(s))


def _codes(x, s, fmt):
    """The fp8 values (as torch's fp8 type) of x / s, to nearest even, saturating."""
    return (x.float() / s).clamp(-FMAX[fmt], FMAX[fmt]).to(F8[fmt])


def _value(x, fmt):
    """What the fp8 copy of x stands for, in 64 bits."""
    _, s = _scale(x, fmt)
    return _codes(x, s, fmt).double() * s.double()


def _exact_backward(x, w, dy):
    g = _value(dy, "e5m2")
    return {"dx": g @ _value(w, "e4m3"), "dw": g.t() @ _value(x, "e4m3"), "db": dy.double().sum(0)}


def _exact_optimizer(case, seed):
    a = _optimizer_inputs(case, seed)
    norm = math.sqrt(sum(float((g * g).double().sum()) for g in a["g"]))
    factor = CLIP / norm if norm > CLIP else 1.0
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    lr, eps = float(np.float32(LR)), float(np.float32(EPS))

    def one(i):
        g = a["g"][i].double() * factor
        m = b1 * a["m"][i].double() + (1 - b1) * g
        v = b2 * a["v"][i].double() + (1 - b2) * g * g
        return a["p"][i].double() - lr * (m / (1 - b1 ** STEP)) / ((v / (1 - b2 ** STEP)).sqrt() + eps), m, v

    w = [i for i, p in enumerate(a["p"]) if p.dim() == 2]
    every = [one(i)[0].abs().max() for i in range(len(a["p"]))]
    ends = [one(w[0]), one(w[-1])]
    return {"norm": torch.tensor([norm], dtype=torch.float64), "absmax": torch.stack(every),
            "scale": torch.stack([every[i] / 448.0 for i in w]), "p": [e[0] for e in ends],
            "m": [e[1] for e in ends], "v": [e[2] for e in ends], "b": one(len(a["p"]) - 1)[0], "q": [None, None],
            "qt": [None, None]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        got = {k: [] for k in (("y", "dx", "dw", "db") if case["backward"] else ("y",))}
        for a in _model_inputs(case, seed):
            got["y"].append(_value(a["x"], "e4m3") @ _value(a["w"], "e4m3").t() + a["b"].double())
            if case["backward"]:
                for k, v in _exact_backward(a["x"], a["w"], a["dy"]).items():
                    got[k].append(v)
        return got
    if kind == "backward":
        a = _backward_inputs(case, seed)
        return _exact_backward(a["x"], a["w"], a["dy"])
    if kind == "mlp":
        a = _mlp_inputs(case, seed)
        y1 = _value(a["x"], "e4m3") @ _value(a["w1"], "e4m3").t() + a["b1"].double()
        y = y1.to(torch.bfloat16)  # fc1's output is held in bf16
        return {"y1": y1, "y2": _value(y, "e4m3") @ _value(a["w2"], "e4m3").t() + a["b2"].double()}
    if kind == "convert":
        x, fmt = _convert_input(case, seed), case["fmt"]
        am, s = _scale(x, fmt)
        q = _codes(x, s, fmt)
        return {"absmax": am.double().reshape(1), "scale": s.double().reshape(1), "codes": None,
                "back": q.double() * s.double()}
    if kind == "layernorm":
        a = _layernorm_inputs(case, seed)
        x = a["x"].double()
        y = (x - x.mean(1, keepdim=True)) / (x.var(1, unbiased=False, keepdim=True) + 1e-5).sqrt()
        y = (y * a["gamma"].double() + a["beta"].double()).to(a["x"].dtype)
        return {"q": None, "qt": None, "scale": _scale(y, "e4m3")[1].double().reshape(1)}
    return _exact_optimizer(case, seed)
