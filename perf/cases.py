"""The work that users of grxBLAS and grxDNN have the libraries do, as cases
that can be prepared, run, counted and checked.

Every case goes through the public entry points (the ctypes binding of the C
API in grxcp_amd) on torch tensors that are already on the GPU, with one
library handle kept for the process. Tensors are written the way torch holds
them (row-major); a row-major matrix [r, c] is a column-major c x r one with
leading dimension c, which is how a torch program calls a BLAS.

Kinds (the fields beside "kind" are the sizes and options):

  gemm   grxblasGemmEx / GemmStridedBatchedEx / GemmExDequant: 16-bit and int8
         products, every layout, one problem or a strided batch
  sgemm  grxblasSgemm / SgemmStridedBatched
  lsq    the gradient of a least-squares fit: r = A x - b, g = s A^T r
         (grxblasSgemv both ways, grxblasSaxpy, grxblasSscal)
  mlp    a transformer's feed-forward half: norm, up projection, GELU, down
         projection added to the residual stream
  attn   grxdnnAttentionForward
  rows   one of the row operations: the norms, softmax, GELU
"""
import ctypes
import math

import torch

import grxcp_amd as g

TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "i8": torch.int8,
         "i32": torch.int32}
GRX = {"bf16": g.GRX_R_16BF, "f16": g.GRX_R_16F, "f32": g.GRX_R_32F, "i8": g.GRX_R_8I,
       "i32": g.GRX_R_32I}
SIZE = {"bf16": 2, "f16": 2, "f32": 4, "i8": 1, "i32": 4}
EPS = 1e-6


def listed():
    return [
        # A large training or prefill product, weights [out, in]: the layout
        # (T, N) that a torch linear layer gives.
        dict(name="gemm_bf16_8192", kind="gemm", dtype="bf16", out="bf16", ta=True, tb=False,
             m=8192, n=8192, k=8192, batch=1),
        # A quantised projection: int8 activations and weights, per-channel scales.
        dict(name="gemm_i8_dequant", kind="gemm", dtype="i8", out="deq", ta=True, tb=False,
             m=4096, n=28672, k=8192, batch=1),
        # An ordinary product of two column-major matrices (N, N) of odd sizes, fp32 result.
        dict(name="gemm_f16_nn_odd", kind="gemm", dtype="f16", out="f32", ta=False, tb=False,
             m=1999, n=1537, k=2301, batch=1),
        # Many small products at once: per-head attention scores.
        dict(name="gemm_bf16_batched", kind="gemm", dtype="bf16", out="bf16", ta=True, tb=False,
             m=256, n=256, k=128, batch=64),
        # A feed-forward block in decoding: 16 sequences, one token each.
        dict(name="mlp_decode", kind="mlp", dtype="bf16", norm="rms", act="tanh", tokens=16,
             hidden=4096, inner=16384),
        # The smallest fp32 product that the benchmark has.
        dict(name="sgemm_512", kind="sgemm", ta=False, tb=False, m=512, n=512, k=512, batch=1),
        # fp32 of odd sizes, the second operand transposed.
        dict(name="sgemm_nt_odd", kind="sgemm", ta=False, tb=True, m=2001, n=1537, k=1023, batch=1),
        # Level 1 and 2: matrix times vector forward and backward.
        dict(name="lsq_gradient", kind="lsq", m=8192, n=4096),
        # Causal attention of a long prefill.
        dict(name="attn_causal_4096", kind="attn", dtype="bf16", causal=True, packed=False,
             b=4, h=32, s=4096, d=128),
        # Full attention of an encoder: a packed QKV buffer, a length that is no tile's multiple.
        dict(name="attn_full_1000", kind="attn", dtype="f16", causal=False, packed=True,
             b=2, h=16, s=1000, d=64),
        # A norm over a long prefill.
        dict(name="rmsnorm_8192", kind="rows", op="rms", dtype="bf16", rows=16384, hidden=8192),
        # Probabilities over a vocabulary of odd size, fp32 as the logits are.
        dict(name="softmax_vocab", kind="rows", op="softmax", dtype="f32", rows=2048, hidden=32001),
    ]


def _log(rng, lo, hi, step=1):
    """A size between lo and hi, even over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choice(["large", "odd", "decode", "i8", "batched", "mlp", "sgemm", "sgemm", "lsq",
                       "attn", "attn", "rows", "rows", "rows"])
    half = rng.choice(["bf16", "f16"])
    if kind == "large":
        while True:
            c = dict(kind="gemm", dtype=half, out=half, ta=rng.random() < 0.7, tb=rng.random() < 0.3,
                     m=_log(rng, 1024, 8192, 64), n=_log(rng, 1024, 8192, 64),
                     k=_log(rng, 1024, 8192, 64), batch=1)
            if c["m"] * c["n"] * c["k"] <= 2 ** 38:
                return c
    if kind == "odd":
        return dict(kind="gemm", dtype=half, out=rng.choice([half, "f32"]), ta=rng.random() < 0.5,
                    tb=rng.random() < 0.5, m=_log(rng, 64, 3000), n=_log(rng, 64, 3000),
                    k=_log(rng, 64, 3000), batch=1)
    if kind == "decode":
        return dict(kind="gemm", dtype=half, out=rng.choice([half, "f32"]), ta=True, tb=False,
                    m=_log(rng, 1024, 16384, 64), n=_log(rng, 1, 128),
                    k=_log(rng, 1024, 16384, 64), batch=1)
    if kind == "i8":
        return dict(kind="gemm", dtype="i8", out=rng.choice(["deq", "i32"]), ta=True, tb=False,
                    m=_log(rng, 256, 4096, rng.choice([1, 64])),
                    n=_log(rng, 16, 8192, rng.choice([1, 64])),
                    k=_log(rng, 512, 8192, 16), batch=1)
    if kind == "batched":
        # scores (T, N) or weighted values (N, N) of attention done with products
        e = _log(rng, 64, 512, rng.choice([1, 64]))
        d = rng.choice([64, 128])
        ta = rng.random() < 0.5
        return dict(kind="gemm", dtype=half, out=half, ta=ta, tb=False, m=e if ta else d, n=e,
                    k=d if ta else e, batch=_log(rng, 8, 256))
    if kind == "mlp":
        hidden = _log(rng, 768, 4096, 64)
        return dict(kind="mlp", dtype=half, norm=rng.choice(["rms", "layer"]),
                    act=rng.choice(["tanh", "erf"]), tokens=_log(rng, 1, 2048), hidden=hidden,
                    inner=4 * hidden)
    if kind == "sgemm":
        batch = rng.choice([1, 1, 1, 8])
        top = 2048 if batch == 1 else 512
        step = rng.choice([1, 1, 16])
        return dict(kind="sgemm", ta=rng.random() < 0.4, tb=rng.random() < 0.4,
                    m=_log(rng, 64, top, step), n=_log(rng, 64, top, step),
                    k=_log(rng, 64, top, step), batch=batch)
    if kind == "lsq":
        return dict(kind="lsq", m=_log(rng, 100, 16384), n=_log(rng, 100, 8192))
    if kind == "attn":
        while True:
            c = dict(kind="attn", dtype=half, causal=rng.random() < 0.6, packed=rng.random() < 0.5,
                     b=_log(rng, 1, 8), h=_log(rng, 4, 32, 4), s=_log(rng, 64, 4096),
                     d=rng.choice([64, 128]))
            if work(c)["flops"] <= 4e11:
                return c
    op = rng.choice(["rms", "layer", "softmax", "erf", "tanh"])
    dtype = rng.choice(["bf16", "f16", "f32"])
    while True:
        hidden = _log(rng, 64, 65536, rng.choice([1, 8, 64]))
        c = dict(kind="rows", op=op, dtype=dtype, rows=_log(rng, 1, 16384), hidden=min(hidden, 65536))
        if c["rows"] * c["hidden"] <= 2 ** 26:
            return c


# ---- preparing -------------------------------------------------------------

class _Lib:
    """The process's library handles, on the stream that torch uses."""
    blas = None
    dnn = None

    @classmethod
    def get(cls):
        if cls.blas is None:
            cls.blas, cls.dnn = g.Blas(), g.Dnn()
            stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            cls.blas.set_stream(stream)
            cls.dnn.set_stream(stream)
        return cls


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


class _Rand:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, dtype, scale=1.0):
        x = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return x.mul_(scale).to(TORCH[dtype])

    def int8(self, shape):
        return torch.randint(-127, 128, shape, generator=self.gen, device="cuda", dtype=torch.int8)

    def uniform(self, shape, lo, hi):
        x = torch.rand(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return x.mul_(hi - lo).add_(lo)


def _inputs(case, seed):
    """The input tensors of a case, from the seed alone."""
    r, kind = _Rand(seed), case["kind"]
    if kind in ("gemm", "sgemm"):
        m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
        # column-major storage, so torch sees the transposed shape
        sa = (batch, m, k) if case["ta"] else (batch, k, m)
        sb = (batch, k, n) if case["tb"] else (batch, n, k)
        dtype = case.get("dtype", "f32")
        if dtype == "i8":
            x = dict(a=r.int8(sa), b=r.int8(sb))
            if case["out"] == "deq":
                x["scale"] = r.uniform((n,), 0.0005, 0.005)
            return x
        return dict(a=r.normal(sa, dtype, k ** -0.5), b=r.normal(sb, dtype))
    if kind == "lsq":
        m, n = case["m"], case["n"]
        return dict(a=r.normal((n, m), "f32", n ** -0.5), x=r.normal((n,), "f32"), b=r.normal((m,), "f32"))
    if kind == "mlp":
        t, d, f, dt = case["tokens"], case["hidden"], case["inner"], case["dtype"]
        return dict(x=r.normal((t, d), dt), gamma=(1 + r.normal((d,), "f32", 0.1)).to(TORCH[dt]),
                    beta=r.normal((d,), dt, 0.1), up=r.normal((f, d), dt, d ** -0.5),
                    down=r.normal((d, f), dt, f ** -0.5))
    if kind == "attn":
        b, h, s, d = case["b"], case["h"], case["s"], case["d"]
        shape = (b, s, 3, h, d) if case["packed"] else (3, b, h, s, d)
        return dict(qkv=r.normal(shape, case["dtype"]))
    rows, hidden, dt = case["rows"], case["hidden"], case["dtype"]
    x = dict(x=r.normal((rows, hidden), dt, 2.0 if case["op"] == "softmax" else 1.0))
    if case["op"] in ("rms", "layer"):
        x["gamma"] = (1 + r.normal((hidden,), "f32", 0.1)).to(TORCH[dt])
        x["beta"] = r.normal((hidden,), dt, 0.1)
    return x


def _gelu_mode(name):
    return {"erf": g.GELU_ERF, "tanh": g.GELU_TANH}[name]


def prepare(case, seed):
    s, kind = dict(case, **_inputs(case, seed)), case["kind"]
    s["lib"] = _Lib.get()

    def empty(shape, dtype):
        return torch.empty(shape, device="cuda", dtype=TORCH[dtype])

    if kind == "gemm":
        out = {"deq": "bf16"}.get(case["out"], case["out"])
        s["c"] = empty((case["batch"], case["n"], case["m"]), out)
        s["ctype"] = GRX[out]
    elif kind == "sgemm":
        s["c"] = empty((case["batch"], case["n"], case["m"]), "f32")
    elif kind == "lsq":
        s["r"], s["grad"] = empty((case["m"],), "f32"), empty((case["n"],), "f32")
    elif kind == "mlp":
        t, d, f, dt = case["tokens"], case["hidden"], case["inner"], case["dtype"]
        s["h"], s["u"], s["y"] = empty((t, d), dt), empty((t, f), dt), empty((t, d), dt)
        s["act_d"], s["inner_d"] = g.TensorDesc(GRX[dt], [t, d]), g.TensorDesc(GRX[dt], [t, f])
        s["w_d"] = g.TensorDesc(GRX[dt], [d])
    elif kind == "attn":
        b, h, n, d, t = case["b"], case["h"], case["s"], case["d"], GRX[case["dtype"]]
        if case["packed"]:
            s["o"] = empty((b, n, h, d), case["dtype"])
            s["in_d"] = g.TensorDesc(t, [b, h, n, d], [n * 3 * h * d, d, 3 * h * d, 1])
            s["out_d"] = g.TensorDesc(t, [b, h, n, d], [n * h * d, d, h * d, 1])
            s["q"], s["k"], s["v"] = (s["qkv"][:, :, i] for i in range(3))
        else:
            s["o"] = empty((b, h, n, d), case["dtype"])
            s["in_d"] = s["out_d"] = g.TensorDesc(t, [b, h, n, d])
            s["q"], s["k"], s["v"] = s["qkv"].unbind(0)
        s["attn_d"] = g.AttnDesc(case["causal"], d ** -0.5)
    else:
        s["y"] = torch.empty_like(s["x"])
        s["x_d"] = g.TensorDesc(GRX[case["dtype"]], [case["rows"], case["hidden"]])
        s["w_d"] = g.TensorDesc(GRX[case["dtype"]], [case["hidden"]])
    return s


# ---- running ---------------------------------------------------------------

def run(s):
    kind, blas, dnn = s["kind"], s["lib"].blas, s["lib"].dnn
    if kind in ("gemm", "sgemm"):
        m, n, k, batch, ta, tb = s["m"], s["n"], s["k"], s["batch"], s["ta"], s["tb"]
        a, b, c = _p(s["a"]), _p(s["b"]), _p(s["c"])
        lda, ldb = k if ta else m, n if tb else k
        if kind == "sgemm" and batch == 1:
            g.check(blas.sgemm(ta, tb, m, n, k, 1.0, a, lda, b, ldb, 0.0, c, m))
        elif kind == "sgemm":
            g.check(blas.sgemm_strided_batched(ta, tb, m, n, k, 1.0, a, lda, m * k, b, ldb, n * k,
                                               0.0, c, m, m * n, batch))
        else:
            t = GRX[s["dtype"]]
            if s["out"] == "deq":
                g.check(blas.gemm_ex_dequant(ta, tb, m, n, k, a, t, lda, b, t, ldb, _p(s["scale"]),
                                             c, s["ctype"], m))
            elif batch == 1:
                g.check(blas.gemm_ex(ta, tb, m, n, k, 1.0, a, t, lda, b, t, ldb, 0.0, c,
                                     s["ctype"], m))
            else:
                g.check(blas.gemm_strided_batched_ex(ta, tb, m, n, k, 1.0, a, t, lda, m * k, b, t,
                                                     ldb, n * k, 0.0, c, s["ctype"], m, m * n,
                                                     batch))
        return s["c"]
    if kind == "lsq":
        m, n, L, h = s["m"], s["n"], blas.L, blas.h
        a, x, r, grad = _p(s["a"]), _p(s["x"]), _p(s["r"]), _p(s["grad"])
        one, zero = g.fptr(1.0), g.fptr(0.0)
        g.check(L.grxblasSgemv(h, g.OP_N, m, n, one, a, m, x, 1, zero, r, 1))
        g.check(L.grxblasSaxpy(h, m, g.fptr(-1.0), _p(s["b"]), 1, r, 1))
        g.check(L.grxblasSgemv(h, g.OP_T, m, n, one, a, m, r, 1, zero, grad, 1))
        g.check(L.grxblasSscal(h, n, g.fptr(2.0 / m), grad, 1))
        return [s["r"], s["grad"]]
    if kind == "mlp":
        t, d, f, dt = s["tokens"], s["hidden"], s["inner"], GRX[s["dtype"]]
        x, h, u, y = _p(s["x"]), _p(s["h"]), _p(s["u"]), _p(s["y"])
        if s["norm"] == "rms":
            g.check(dnn.rmsnorm(s["act_d"], x, s["w_d"], _p(s["gamma"]), EPS, s["act_d"], h))
        else:
            g.check(dnn.layernorm(s["act_d"], x, s["w_d"], _p(s["gamma"]), _p(s["beta"]), EPS,
                                  s["act_d"], h))
        g.check(blas.gemm_ex(1, 0, f, t, d, 1.0, _p(s["up"]), dt, d, h, dt, d, 0.0, u, dt, f))
        g.check(dnn.gelu(_gelu_mode(s["act"]), s["inner_d"], u, s["inner_d"], u))
        s["y"].copy_(s["x"])
        g.check(blas.gemm_ex(1, 0, d, t, f, 1.0, _p(s["down"]), dt, f, u, dt, f, 1.0, y, dt, d))
        return [s["h"], s["u"], s["y"]]
    if kind == "attn":
        g.check(dnn.attention(s["attn_d"], s["in_d"], _p(s["q"]), s["in_d"], _p(s["k"]), s["in_d"],
                              _p(s["v"]), s["out_d"], _p(s["o"])))
        return s["o"]
    x, y, op = _p(s["x"]), _p(s["y"]), s["op"]
    if op == "rms":
        g.check(dnn.rmsnorm(s["x_d"], x, s["w_d"], _p(s["gamma"]), EPS, s["x_d"], y))
    elif op == "layer":
        g.check(dnn.layernorm(s["x_d"], x, s["w_d"], _p(s["gamma"]), _p(s["beta"]), EPS, s["x_d"], y))
    elif op == "softmax":
        g.check(dnn.softmax(s["x_d"], x, s["x_d"], y))
    else:
        g.check(dnn.gelu(_gelu_mode(op), s["x_d"], x, s["x_d"], y))
    return s["y"]


# ---- counting --------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("gemm", "sgemm"):
        m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
        i = SIZE[case.get("dtype", "f32")]
        o = {"deq": 2}.get(case.get("out", "f32")) or SIZE[case.get("out", "f32")]
        extra = 4 * n if case.get("out") == "deq" else 0
        return {"bytes": batch * (i * (m * k + n * k) + o * m * n) + extra,
                "flops": 2.0 * batch * m * n * k}
    if kind == "lsq":
        # A is read for each direction; r is the first one's result and the second one's input
        m, n = case["m"], case["n"]
        return {"bytes": 4 * (2 * m * n + 3 * m + 2 * n), "flops": 4.0 * m * n + 2 * m + n}
    if kind == "mlp":
        t, d, f = case["tokens"], case["hidden"], case["inner"]
        # weights, x, gamma, beta, and the three results
        return {"bytes": 2 * (2 * d * f + 3 * t * d + t * f + 2 * d), "flops": 4.0 * t * d * f}
    if kind == "attn":
        b, h, s, d = case["b"], case["h"], case["s"], case["d"]
        pairs = s * (s + 1) // 2 if case["causal"] else s * s
        return {"bytes": 2 * 4 * b * h * s * d, "flops": 4.0 * b * h * d * pairs}
    n = case["rows"] * case["hidden"]
    per = {"rms": 4, "layer": 7, "softmax": 5, "erf": 20, "tanh": 10}[case["op"]]
    return {"bytes": 2 * n * SIZE[case["dtype"]], "flops": float(per * n)}


def tolerance(case):
    kind = case["kind"]
    if kind == "gemm" and case["dtype"] == "i8":
        return "exact"                      # whole sums; the scaled result's bits are defined too
    if kind in ("sgemm", "lsq") or (kind == "gemm" and case["out"] == "f32"):
        return {"rel": 4e-6}                # fp32 sums in another order
    if kind == "rows" and case["dtype"] == "f32":
        return {"rel": 1e-6}
    if kind == "mlp":
        # an input of each stage is the 16-bit result of the one before
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
    # one rounding to 16 bits (attention: also of the probabilities)
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3}


# ---- the same in 64 bits ----------------------------------------------------

def _gelu64(x, act):
    if act == "erf":
        return 0.5 * x * torch.special.erfc(-x / math.sqrt(2.0))
    return x * torch.sigmoid(2 * math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3))


def _norm64(x, gamma, beta, layer):
    if layer:
        x = x - x.mean(-1, keepdim=True)
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma
    return x + beta if layer else x


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind in ("gemm", "sgemm"):
        c = []
        for i in range(case["batch"]):
            # C^T [n, m] = op(B)^T op(A)^T
            a, b = s["a"][i].double(), s["b"][i].double()
            at = a.t().contiguous() if case["ta"] else a
            bt = b.t().contiguous() if case["tb"] else b
            c.append(bt @ at)
        c = torch.stack(c)
        if case.get("out") == "deq":
            return c * s["scale"].double()[None, :, None]
        return c.round().to(torch.int32) if case.get("out") == "i32" else c
    if kind == "lsq":
        a = s["a"].double()                  # [n, m]
        r = s["x"].double() @ a - s["b"].double()
        return [r, (a @ r) * (2.0 / case["m"])]
    if kind == "mlp":
        x = s["x"].double()
        h = _norm64(x, s["gamma"].double(), s["beta"].double(), case["norm"] == "layer")
        u = _gelu64(h @ s["up"].double().t().contiguous(), case["act"])
        return [h, u, x + u @ s["down"].double().t().contiguous()]
    if kind == "attn":
        qkv = s["qkv"].permute(2, 0, 3, 1, 4) if case["packed"] else s["qkv"]
        b, h, n, d = case["b"], case["h"], case["s"], case["d"]
        o = torch.empty((b, h, n, d), device="cuda", dtype=torch.float64)
        mask = torch.ones((n, n), device="cuda", dtype=torch.bool).triu(1) if case["causal"] else None
        for i in range(b):
            for j in range(h):
                q, k, v = (qkv[t, i, j].double() for t in range(3))
                w = (q @ k.t().contiguous()) * d ** -0.5
                if mask is not None:
                    w = w.masked_fill_(mask, -math.inf)
                o[i, j] = torch.softmax(w, -1) @ v
        return o.permute(0, 2, 1, 3).contiguous() if case["packed"] else o
    x, op = s["x"].double(), case["op"]
    if op in ("rms", "layer"):
        return _norm64(x, s["gamma"].double(), s["beta"].double(), op == "layer")
    return torch.softmax(x, -1) if op == "softmax" else _gelu64(x, op)
