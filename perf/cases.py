"""The work this library is timed on: its operators and plans as a program
calls them, over the range of sizes, data types and directions in use.

Each case names a kind (one of the functions below) and its sizes.  The
kinds are the layers of the BW++ programs (`plans/`), each through the
operator entry points, and one whole program through the plan executor:

  rows       the row operators of one activation: softmax, LayerNorm,
             RMSNorm, reduce_max with its index and its one-hot gradient
  grads      the bandwidth-bound operators of an autodiff graph: RMSNorm and
             softmax gradients, SiLU gradient, bias add and bias gradient
             (a sum over rows), and a reduce_max over rows with its gradient
  linear     Y = SiLU(X W + b), the forward of one layer
  linear_bwd the three products of a linear layer in training: Y = X W + b,
             dX = dY W^T, dW = X^T dY
  attention  the attention forward alone (prefill with causal = 1, an
             encoder with causal = 0, decoding where the queries are few
             and the keys are the cache)
  attention_train  the forward that saves lse, then the backward
  block      one transformer block's forward and backward through its
             lowered plan
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "bluewolf-plus-plus_amd"))

import bwpp  # noqa: E402
from bwpp.plan import Plan, load_text  # noqa: E402

_BACKEND = None


def _backend():
    """The handle a program keeps for its lifetime, on torch's stream."""
    global _BACKEND
    if _BACKEND is None:
        _BACKEND = bwpp.HipBackend(0)
    _BACKEND.set_stream(torch.cuda.current_stream())
    return _BACKEND


# ------------------------------------------------------------------- cases


def listed():
    return [
        # The bandwidth-bound operators on a full batch of activations
        # (8192 tokens of width 4096): the benchmark's headline shape.
        dict(name="rows_8192x4096", kind="rows", rows=8192, cols=4096, pad=0),
        # The same on a batch whose row length no vector width divides (an
        # odd class count): rows that start at any 4-byte address.
        dict(name="rows_2047x5003", kind="rows", rows=2047, cols=5003, pad=0),
        # What autodiff adds around the matrix products of a training step,
        # on 4096 tokens of width 4096.
        dict(name="grads_4096x4096", kind="grads", rows=4096, cols=4096, pad=0),
        # A prefill's widest layer: bf16 MLP up-projection of 4096 tokens.
        dict(name="linear_bf16_4096x4096x11008", kind="linear", dtype="bf16", M=4096, K=4096, N=11008),
        # The same layer while decoding: a few tokens against all weights.
        dict(name="linear_bf16_16x4096x11008", kind="linear", dtype="bf16", M=16, K=4096, N=11008),
        # The smallest call in use: the fp32 product of the reference's
        # benchmark default, where launches and latency count.
        dict(name="linear_f32_256", kind="linear", dtype="f32", M=256, K=256, N=256),
        # Training a layer on a ragged batch in bf16: a token count and a
        # width that no tile divides, forward and both gradients.
        dict(name="linear_bwd_bf16_1337x1024x3000", kind="linear_bwd", dtype="bf16", M=1337, K=1024, N=3000),
        # The same in fp32 with odd sizes (rows at any 4-byte address).
        dict(name="linear_bwd_f32_777x1021x2043", kind="linear_bwd", dtype="f32", M=777, K=1021, N=2043),
        # Long-sequence causal training in bf16 with head dim 128.
        dict(name="attn_train_bf16_d128_8x32x2048", kind="attention_train", dtype="bf16", B=8, H=32, M=2048, N=2048,
             d=128, causal=1),
        # The smaller head dim on a ragged sequence length.
        dict(name="attn_train_bf16_d64_4x16x1000", kind="attention_train", dtype="bf16", B=4, H=16, M=1000, N=1000,
             d=64, causal=1),
        # One decoding step: a query per sequence against a long cache.
        dict(name="attn_decode_bf16_d128_8x32x4095", kind="attention", dtype="bf16", B=8, H=32, M=1, N=4095, d=128,
             causal=1),
        # A whole training step of a transformer block (fp32, 8 sequences
        # of 512 tokens, width 1024, 16 heads, MLP 4096).
        dict(name="block_train_f32_8x512x1024", kind="block", B=8, T=512, D=1024, heads=16, F=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """Half of the sizes are the multiples that networks are built with, the
    other half any number of the range."""
    n = _log_int(rng, lo, hi)
    if rng.random() < 0.5:
        n = min(hi, max(lo, (n + step - 1) // step * step))
    return n


def draw(rng):
    kind = rng.choice(["rows", "rows", "grads", "linear", "linear", "linear_bwd", "linear_bwd", "attention",
                       "attention", "attention_train", "attention_train", "block"])
    if kind in ("rows", "grads"):
        cols = _size(rng, 64, 16384 if kind == "rows" else 8192, 64)
        top = min(32768, 8192 * 4096 // cols) if kind == "rows" else min(8192, 4096 * 4096 // cols)
        rows = _log_int(rng, 1, top)
        return dict(kind=kind, rows=rows, cols=cols, pad=rng.choice([0, 0, 0, 1, 4]))
    if kind == "linear":
        K, N = _size(rng, 64, 8192, 64), _size(rng, 64, 11008, 64)
        dtype = rng.choice(["bf16", "bf16", "f32"])
        # a prompt, a batch of decoding sequences, or anything between; fp32
        # runs an order of magnitude slower and gets the smaller products
        top = min(4096, (4096 * 4096 * 11008 if dtype == "bf16" else 2048 ** 3) // (K * N))
        return dict(kind=kind, dtype=dtype, M=_size(rng, 1, max(1, top), 32), K=K, N=N)
    if kind == "linear_bwd":
        dtype = rng.choice(["bf16", "f32"])
        K, N = _size(rng, 64, 4096, 64), _size(rng, 64, 4096, 64)
        top = min(4096, (4096 * 4096 * 2048 if dtype == "bf16" else 1024 ** 3) // (K * N))
        return dict(kind=kind, dtype=dtype, M=_size(rng, 32, max(32, top), 32), K=K, N=N)
    if kind == "attention":
        dtype, d, B, H = rng.choice(["bf16", "bf16", "f32"]), rng.choice([64, 128]), rng.randint(1, 16), rng.choice(
            [4, 8, 16, 32])
        if rng.random() < 0.6:  # decoding: few queries, a long cache
            top = min(8192, 8 * 32 * 4096 * 128 // (B * H * d))
            N = _log_int(rng, 64, max(64, top))
            return dict(kind=kind, dtype=dtype, B=B, H=H, M=rng.choice([1, 1, 1, 4, 16]), N=N, d=d, causal=1)
        top = int(math.sqrt((2 ** 36 if dtype == "bf16" else 2 ** 33) / (B * H * d)))
        S = _size(rng, 33, max(33, min(4096, top)), 64)
        return dict(kind=kind, dtype=dtype, B=B, H=H, M=S, N=S, d=d, causal=rng.choice([0, 1]))
    if kind == "attention_train":
        dtype, d, B, H = rng.choice(["bf16", "bf16", "f32"]), rng.choice([64, 64, 128, 96]), rng.randint(
            1, 8), rng.choice([4, 8, 16])
        # a head dim outside 64 / 128 is for small models
        budget = 2 ** 28 if d == 96 else 2 ** 34 if dtype == "bf16" else 2 ** 31
        S = _size(rng, 33, max(33, min(2048, int(math.sqrt(budget / (B * H * d))))), 64)
        return dict(kind=kind, dtype=dtype, B=B, H=H, M=S, N=S, d=d, causal=rng.choice([0, 1]))
    D = rng.choice([256, 512, 1024])
    B = rng.randint(1, 8)
    return dict(kind="block", B=B, T=_size(rng, 33, 512, 64), D=D, heads=D // 64, F=4 * D)


# ------------------------------------------------------------------ inputs


class _Inputs:
    """Seeded draws on the GPU; the same (seed, order) gives the same values."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(std).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo)


_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "bf16": 2}
_CODE = {"f32": int(bwpp.DType.F32), "bf16": int(bwpp.DType.BF16)}
EPS = 1e-5


def _inputs(case, seed):
    """The tensors a pass reads, by name."""
    r = _Inputs(seed)
    k = case["kind"]
    if k in ("rows", "grads"):
        rows, cols, ld = case["rows"], case["cols"], case["cols"] + case["pad"]
        t = dict(x=r.normal(rows, ld), gamma=r.uniform(cols, lo=0.5, hi=1.5), beta=r.normal(cols, std=0.1))
        if k == "rows":
            t["dy"] = r.normal(rows)
        else:
            t["dy"] = r.normal(rows, ld)
            t["p"] = torch.zeros(rows, ld, device="cuda")  # the forward's probabilities
            t["p"][:, :cols] = torch.softmax(r.normal(rows, cols), dim=1)
            t["dcol"] = r.normal(cols)
        return t
    if k in ("linear", "linear_bwd"):
        M, K, N, dt = case["M"], case["K"], case["N"], _TORCH[case["dtype"]]
        t = dict(x=r.normal(M, K, dtype=dt), w=r.normal(K, N, std=0.02, dtype=dt), b=r.normal(N, std=0.02, dtype=dt))
        if k == "linear_bwd":
            t["dy"] = r.normal(M, N, std=0.1, dtype=dt)
        return t
    if k in ("attention", "attention_train"):
        B, H, M, N, d, dt = (case[i] for i in ("B", "H", "M", "N", "d", "dtype"))
        dt = _TORCH[dt]
        t = dict(q=r.normal(B, H, M, d, dtype=dt), k=r.normal(B, H, N, d, dtype=dt), v=r.normal(B, H, N, d, dtype=dt))
        if k == "attention_train":
            t["do"] = r.normal(B, H, M, d, dtype=dt)
        return t
    BT, D, F = case["B"] * case["T"], case["D"], case["F"]
    t = dict(x=r.normal(BT, D), g1=r.uniform(D, lo=0.5, hi=1.5), g2=r.uniform(D, lo=0.5, hi=1.5))
    for n in ("wq", "wk", "wv", "wo"):
        t[n] = r.normal(D, D, std=0.02)
    t["w1"], t["w2"] = r.normal(D, F, std=0.02), r.normal(F, D, std=0.02)
    return t


class _Device:
    """A plan value's device memory (float32), for torch to wrap."""

    def __init__(self, plan, name, shape):
        self.__cuda_array_interface__ = dict(data=(plan.ptr(name), False), shape=tuple(shape), typestr="<f4",
                                             version=2)


def _value(plan, name, shape):
    """A plan value as a tensor over the plan's own memory, which lives as
    long as the plan: the tensor keeps it."""
    t = torch.as_tensor(_Device(plan, name, shape), device="cuda")
    t.plan = plan
    return t


_BLOCK_OUTPUTS = ("out", "loss", "dx", "dg1", "dg2", "dwq", "dwk", "dwv", "dwo", "dw1", "dw2")


def _block_shapes(case):
    BT, D, F = case["B"] * case["T"], case["D"], case["F"]
    return dict(out=(BT, D), loss=(1,), dx=(BT, D), dg1=(D,), dg2=(D,), dwq=(D, D), dwk=(D, D), dwv=(D, D),
                dwo=(D, D), dw1=(D, F), dw2=(F, D))


def prepare(case, seed):
    be = _backend()
    t = _inputs(case, seed)
    k = case["kind"]
    new = lambda *s, dtype=torch.float32: torch.zeros(*s, dtype=dtype, device="cuda")
    st = dict(case=case, be=be, t=t)
    if k == "rows":
        rows, cols, ld = case["rows"], case["cols"], case["cols"] + case["pad"]
        st["out"] = dict(softmax=new(rows, ld), layernorm=new(rows, ld), rmsnorm=new(rows, ld), maxv=new(rows),
                         argmax=new(rows, dtype=torch.int32), dx=new(rows, ld))
        st["p"] = (bwpp.SoftmaxParams(rows, cols, ld), bwpp.RmsnormParams(rows, cols, ld, EPS),
                   bwpp.ReduceParams(rows, cols, ld, 1))
    elif k == "grads":
        rows, cols, ld = case["rows"], case["cols"], case["cols"] + case["pad"]
        st["out"] = dict(dx=new(rows, ld), dgamma=new(cols), dbeta=new(cols), dscore=new(rows, ld), dsilu=new(rows, ld),
                         biased=new(rows, ld), dbias=new(cols), maxv=new(cols), argmax=new(cols, dtype=torch.int32),
                         dmax=new(rows, ld))
        st["p"] = (bwpp.SoftmaxParams(rows, cols, ld), bwpp.RmsnormParams(rows, cols, ld, EPS),
                   bwpp.ReduceParams(rows, cols, ld, 0), bwpp.ElementwiseParams(rows, cols, ld, 0, 1))
    elif k == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        st["out"] = dict(y=new(M, N, dtype=t["x"].dtype))
        st["p"] = bwpp.MatmulParams(M, N, K, K, N, N, _CODE[case["dtype"]], int(bwpp.Epilogue.ADD_SILU), 0, 0)
    elif k == "linear_bwd":
        M, K, N, c = case["M"], case["K"], case["N"], _CODE[case["dtype"]]
        dt = t["x"].dtype
        st["out"] = dict(y=new(M, N, dtype=dt), dx=new(M, K, dtype=dt), dw=new(K, N, dtype=dt))
        st["p"] = (bwpp.MatmulParams(M, N, K, K, N, N, c, int(bwpp.Epilogue.ADD), 0, 0),
                   bwpp.MatmulParams(M, K, N, N, N, K, c, 0, 0, 1),
                   bwpp.MatmulParams(K, N, M, K, N, N, c, 0, 1, 0))
    elif k in ("attention", "attention_train"):
        B, H, M, N, d = (case[i] for i in ("B", "H", "M", "N", "d"))
        st["p"] = bwpp.AttentionParams(M=M, N=N, K=d, D=d, ldq=d, ldk=d, ldv=d, ldo=d, batch=B, heads=H,
                                       scale=d ** -0.5, causal=case["causal"], dtype=_CODE[case["dtype"]])
        st["out"] = dict(o=torch.zeros_like(t["q"]))
        if k == "attention_train":
            st["out"].update(lse=new(B, H, M), dq=torch.zeros_like(t["q"]), dk=torch.zeros_like(t["k"]),
                             dv=torch.zeros_like(t["v"]))
    else:
        st["plan"] = Plan(be, load_text("block_train", BATCH=case["B"], T=case["T"], D=case["D"], H=case["F"],
                                        HEADS=case["heads"]))
        st["plan"].allocate()
        for name, v in t.items():
            st["plan"].bind(name, v)
        st["out"] = {n: _value(st["plan"], n, s) for n, s in _block_shapes(case).items()}
    return st


# --------------------------------------------------------------- one pass


def run(st):
    be, t, o, case = st["be"], st["t"], st["out"], st["case"]
    k = case["kind"]
    if k == "rows":
        sp, rp, mp = st["p"]
        be.dispatch_softmax(t["x"], o["softmax"], sp)
        be.dispatch_layernorm(t["x"], t["gamma"], t["beta"], o["layernorm"], rp)
        be.dispatch_rmsnorm(t["x"], t["gamma"], None, o["rmsnorm"], rp)
        be.dispatch_reduce_max(t["x"], o["maxv"], o["argmax"], mp)
        be.dispatch_reduce_max_grad_argmax(t["x"], None, t["dy"], o["dx"], mp)
    elif k == "grads":
        sp, rp, mp, ep = st["p"]
        be.dispatch_rmsnorm_grad(t["x"], t["gamma"], t["dy"], o["dx"], o["dgamma"], o["dbeta"], rp)
        be.dispatch_softmax_grad(t["p"], t["dy"], o["dscore"], sp)
        be.dispatch_silu_grad(t["x"], t["dy"], o["dsilu"], t["x"].numel())
        be.dispatch_elementwise(t["x"], t["beta"], o["biased"], ep)
        be.dispatch_reduce_sum(t["dy"], o["dbias"], mp)
        be.dispatch_reduce_max(t["x"], o["maxv"], o["argmax"], mp)
        be.dispatch_reduce_max_grad_argmax(None, o["argmax"], t["dcol"], o["dmax"], mp)
    elif k == "linear":
        be.dispatch_matmul(t["x"], t["w"], o["y"], t["b"], st["p"])
    elif k == "linear_bwd":
        fwd, dxp, dwp = st["p"]
        be.dispatch_matmul(t["x"], t["w"], o["y"], t["b"], fwd)
        be.dispatch_matmul(t["dy"], t["w"], o["dx"], None, dxp)
        be.dispatch_matmul(t["x"], t["dy"], o["dw"], None, dwp)
    elif k == "attention":
        be.dispatch_attention(t["q"], t["k"], t["v"], o["o"], st["p"])
    elif k == "attention_train":
        be.dispatch_attention_lse(t["q"], t["k"], t["v"], o["o"], o["lse"], st["p"])
        be.dispatch_attention_grad(t["q"], t["k"], t["v"], o["o"], t["do"], o["lse"], o["dq"], o["dk"], o["dv"],
                                   st["p"])
    else:
        st["plan"].run()
    return o


# ------------------------------------------------------- what it must cost


def work(case):
    k = case["kind"]
    if k == "rows":
        n, rows, cols = case["rows"] * case["cols"], case["rows"], case["cols"]
        # five reads of x, four full outputs; the vectors once each
        return dict(bytes=9 * n * 4 + 3 * cols * 4 + 3 * rows * 4, flops=30 * n)
    if k == "grads":
        n, cols = case["rows"] * case["cols"], case["cols"]
        # rmsnorm 2 + 1, softmax 2 + 1, silu 2 + 1, bias 1 + 1, sum 1, max 1, max gradient 1
        return dict(bytes=14 * n * 4 + 9 * cols * 4, flops=40 * n)
    if k == "linear":
        M, K, N, e = case["M"], case["K"], case["N"], _BYTES[case["dtype"]]
        return dict(bytes=(M * K + K * N + N + M * N) * e, flops=2.0 * M * K * N)
    if k == "linear_bwd":
        M, K, N, e = case["M"], case["K"], case["N"], _BYTES[case["dtype"]]
        return dict(bytes=(3 * (M * K + K * N + M * N) + N) * e, flops=6.0 * M * K * N)
    if k in ("attention", "attention_train"):
        B, H, M, N, d, e = case["B"], case["H"], case["M"], case["N"], case["d"], _BYTES[case["dtype"]]
        pairs = M * N
        if case["causal"]:  # key n is seen by query m when n <= m + N - M
            pairs = sum(max(0, m + N - M + 1) for m in range(M))
        rows = B * H * (2 * M + 2 * N) * d * e
        if k == "attention":
            return dict(bytes=rows, flops=4.0 * B * H * pairs * d)
        # forward, then q, k, v, o, do, lse in and dq, dk, dv out
        return dict(bytes=rows + B * H * ((4 * M + 4 * N) * d * e + 2 * M * 4), flops=14.0 * B * H * pairs * d)
    B, T, D, F, h = case["B"], case["T"], case["D"], case["F"], case["heads"]
    gemm = 2.0 * B * T * D * (4 * D + 2 * F)
    attn = 4.0 * B * h * (T * (T + 1) // 2) * (D // h)
    # parameters in and their gradients out, x in, out and dx out
    return dict(bytes=4.0 * (2 * (4 * D * D + 2 * D * F + 2 * D) + 3 * B * T * D), flops=3.0 * gemm + 3.5 * attn)


def tolerance(case):
    """About four times the error against exact() over the declared ranges."""
    k = case["kind"]
    if k in ("rows", "grads"):
        return {"rel": 1e-6, "max": 1e-5}
    if k == "block" or case["dtype"] == "f32":
        return {"rel": 6e-6, "max": 5e-5}
    if k in ("linear", "linear_bwd"):  # the rounding of a bf16 result
        return {"rel": 7e-3, "max": 1.6e-2}
    # bf16 probabilities and score gradients; the largest differences are
    # those of gradients that cancel (the first rows of a causal mask)
    return {"rel": 1e-2, "max": 0.5 if k == "attention_train" else 0.13}


# -------------------------------------------------- the same in 64 bits


def _attention_exact(q, k, v, causal, do=None):
    """One (batch, head) slice in float64: o, lse and, with do, dq, dk, dv."""
    M, N, scale = q.shape[0], k.shape[0], q.shape[1] ** -0.5
    s = (q @ k.t().contiguous()) * scale
    if causal:
        m = torch.arange(M, device="cuda")[:, None]
        s.masked_fill_(torch.arange(N, device="cuda")[None, :] > m + (N - M), -math.inf)
    lse = torch.logsumexp(s, dim=1)
    p = torch.exp(s - lse[:, None])
    o = p @ v
    if do is None:
        return o, lse
    dv = p.t().contiguous() @ do
    ds = p * (do @ v.t().contiguous() - (do * o).sum(dim=1, keepdim=True)) * scale
    return o, lse, ds @ k, ds.t().contiguous() @ q, dv


def _block_exact(t, case):
    B, T, h = case["B"], case["T"], case["heads"]
    p = {n: v.double().requires_grad_(True) for n, v in t.items()}
    rms = lambda a, g: a / torch.sqrt((a * a).mean(dim=1, keepdim=True) + EPS) * g
    split = lambda m: m.reshape(B, T, h, -1).permute(0, 2, 1, 3).contiguous()
    n1 = rms(p["x"], p["g1"])
    q, k, v = split(n1 @ p["wq"]), split(n1 @ p["wk"]), split(n1 @ p["wv"])
    s = (q @ k.transpose(-1, -2).contiguous()) * (q.shape[-1] ** -0.5)
    s = s.masked_fill(~torch.ones(T, T, dtype=torch.bool, device="cuda").tril(), -math.inf)
    ctx = (torch.softmax(s, dim=-1) @ v).permute(0, 2, 1, 3).reshape(B * T, -1)
    x1 = p["x"] + ctx @ p["wo"]
    out = x1 + torch.nn.functional.silu(rms(x1, p["g2"]) @ p["w1"]) @ p["w2"]
    loss = (out * out).mean()
    loss.backward()
    r = dict(out=out.detach(), loss=loss.detach().reshape(1))
    r.update({n: p[n[1:]].grad for n in _BLOCK_OUTPUTS if n not in r})
    return {n: r[n] for n in _block_shapes(case)}


def exact(case, seed):
    t = _inputs(case, seed)
    k = case["kind"]
    if k in ("rows", "grads"):
        rows, cols, ld = case["rows"], case["cols"], case["cols"] + case["pad"]

        def full(v):  # the padding columns stay zero
            r = torch.zeros(rows, ld, dtype=torch.float64, device="cuda")
            r[:, :cols] = v
            return r

        x = t["x"][:, :cols].double()
        g, b = t["gamma"].double(), t["beta"].double()
    if k == "rows":
        mean = x.mean(dim=1, keepdim=True)
        var = ((x - mean) ** 2).mean(dim=1, keepdim=True)
        mv = x.max(dim=1).values
        col = torch.arange(cols, device="cuda")
        am = torch.where(x == mv[:, None], col, cols).min(dim=1).values
        dx = torch.where(col[None, :] == am[:, None], t["dy"].double()[:, None], 0.0)
        return dict(softmax=full(torch.softmax(x, dim=1)), layernorm=full((x - mean) / torch.sqrt(var + EPS) * g + b),
                    rmsnorm=full(x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS) * g), maxv=mv,
                    argmax=am.int(), dx=full(dx))
    if k == "grads":
        dy, p = t["dy"][:, :cols].double(), t["p"][:, :cols].double()
        inv = 1.0 / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS)
        xh = x * inv
        dx = inv * (g * dy - xh * (xh * g * dy).mean(dim=1, keepdim=True))
        xf, df = t["x"].double(), t["dy"].double()  # the SiLU gradient runs over the whole buffer
        s = torch.sigmoid(xf)
        mv = x.max(dim=0).values
        row = torch.arange(rows, device="cuda")
        am = torch.where(x == mv[None, :], row[:, None], rows).min(dim=0).values
        dmax = torch.where(row[:, None] == am[None, :], t["dcol"].double()[None, :], 0.0)
        return dict(dx=full(dx), dgamma=(dy * xh).sum(dim=0), dbeta=dy.sum(dim=0),
                    dscore=full(p * (dy - (dy * p).sum(dim=1, keepdim=True))), dsilu=df * s * (1 + xf * (1 - s)),
                    biased=full(x + b), dbias=dy.sum(dim=0), maxv=mv, argmax=am.int(), dmax=full(dmax))
    if k == "linear":
        z = t["x"].double() @ t["w"].double() + t["b"].double()
        return dict(y=z * torch.sigmoid(z))
    if k == "linear_bwd":
        x, w, b, dy = (t[n].double() for n in ("x", "w", "b", "dy"))
        return dict(y=x @ w + b, dx=dy @ w.t().contiguous(), dw=x.t().contiguous() @ dy)
    if k in ("attention", "attention_train"):
        names = ("o",) if k == "attention" else ("o", "lse", "dq", "dk", "dv")
        out = {n: torch.empty(t["q"].shape[:3] if n == "lse" else t[n[-1] if n != "o" else "q"].shape,
                              dtype=torch.float64, device="cuda") for n in names}
        for b in range(case["B"]):
            for h in range(case["H"]):
                at = lambda n: t[n][b, h].double()
                r = _attention_exact(at("q"), at("k"), at("v"), case["causal"],
                                     at("do") if k == "attention_train" else None)
                for n, v in zip(("o", "lse", "dq", "dk", "dv"), r):
                    if n in out:
                        out[n][b, h] = v
        return out
    return _block_exact(t, case)
