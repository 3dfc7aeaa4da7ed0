"""What a program spends its time on in this library, as cases to measure.

Each case is one pass of a layer or a block through the Python entry points of
``cgadimpl_amd``, as a training step (forward and VJP) or an inference call
runs it.  The kinds:

- ``rmsnorm``      y = x * rsqrt(mean(x^2) + eps) * gamma and its VJP: the layer
                   this library is built around;
- ``rms_mul``      the same layer written ``rms(x) * gamma``, two graph nodes, with
                   the one-pass VJP of the pair;
- ``norm_linear``  RMSNorm followed by a dense bf16 projection, forward and the
                   full VJP (dx, dgamma, dW);
- ``norm_linear_infer``  its forward alone on the few rows of a decoding batch;
- ``linear``       x W^T + b on bf16 with gradients of x, W and b;
- ``matmul_f32``   a product of fp32 matrices with both gradients;
- ``softmax``, ``logsumexp``  row softmax / log-sum-exp of logits and the VJP;
- ``layernorm``    LayerNorm without affine parameters and its VJP;
- ``mul_bcast``    an element-wise product under broadcasting and its VJP.

Sizes are those of the benchmark's configurations, the tests and the benchmark's
wide-row tables, or round numbers of the same ranges.
"""
import math

import torch

import cgadimpl_amd as agk

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
EPS = 1e-6


def listed():
    return [
        # The smallest training call: 4 x 128 tokens of a narrow model.  Latency
        # and launches, not bytes, make its time.
        dict(name="rmsnorm_small", kind="rmsnorm", dtype="f32", rows=512, cols=512),
        # The library's headline: 32 x 2048 tokens, hidden 4096, fp32.
        dict(name="rmsnorm_headline", kind="rmsnorm", dtype="f32", rows=65536, cols=4096),
        # An odd number of rows of a width that is no multiple of a 16-byte slot
        # (a pruned or concatenated hidden size): rows start at every alignment.
        dict(name="rmsnorm_ragged", kind="rmsnorm", dtype="f32", rows=4099, cols=1030),
        # A bf16 layer of an ordinary batch in the two-node form of the graph API.
        dict(name="rms_mul_batch", kind="rms_mul", dtype="bf16", rows=8192, cols=8192),
        # A training step of RMSNorm + up-projection at 8192 tokens.
        dict(name="norm_linear_train", kind="norm_linear", dtype="bf16", rows=8192, cols=4096,
             out=11008),
        # The same block while decoding: 16 sequences, one token each.
        dict(name="norm_linear_decode", kind="norm_linear_infer", dtype="bf16", rows=16, cols=4096,
             out=11008),
        # A projection with a bias at the odd token count of a packed batch.
        dict(name="linear_train", kind="linear", dtype="bf16", rows=1032, cols=4096, out=4096),
        # fp32 matmul of a small model's step.
        dict(name="matmul_f32_train", kind="matmul_f32", dtype="f32", rows=1024, cols=1024,
             out=1024),
        # Softmax over a vocabulary that is a multiple of nothing.
        dict(name="softmax_vocab", kind="softmax", dtype="bf16", rows=8192, cols=50257),
        # The log-sum-exp of a loss head over fp32 logits of a small batch.
        dict(name="logsumexp_head", kind="logsumexp", dtype="f32", rows=1024, cols=50257),
        # LayerNorm of an ordinary batch with an odd number of rows.
        dict(name="layernorm_batch", kind="layernorm", dtype="f32", rows=4099, cols=1000),
        # Per-sequence channel scales over a batch of sequences.
        dict(name="mul_bcast_scale", kind="mul_bcast", dtype="bf16", form="sequence", batch=32,
             rows=2048, cols=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A row width: half of them a multiple of 16 bytes in either type, half anything."""
    w = _log_int(rng, lo, hi)
    return max(8, w // 8 * 8) if rng.random() < 0.5 else w


def draw(rng):
    kind = rng.choice([c["kind"] for c in listed()])
    dtype = rng.choice(["f32", "bf16"])
    if kind in ("rmsnorm", "rms_mul", "layernorm"):
        cols = _width(rng, 64, 16384)
        rows = min(_log_int(rng, 64, 65536), (1 << 28) // cols)
        return dict(kind=kind, dtype=dtype, rows=rows, cols=cols)
    if kind == "norm_linear":
        return dict(kind=kind, dtype="bf16", rows=8 * _log_int(rng, 32, 1024),
                    cols=rng.choice([8, 64]) * _log_int(rng, 16, 64),
                    out=8 * _log_int(rng, 64, 1376))
    if kind == "norm_linear_infer":
        return dict(kind=kind, dtype="bf16", rows=8 * _log_int(rng, 1, 32),
                    cols=rng.choice([8, 64]) * _log_int(rng, 16, 128),
                    out=8 * _log_int(rng, 64, 1376))
    if kind == "linear":
        return dict(kind=kind, dtype="bf16", rows=8 * _log_int(rng, 8, 512),
                    cols=rng.choice([8, 64]) * _log_int(rng, 16, 64),
                    out=8 * _log_int(rng, 64, 1376))
    if kind == "matmul_f32":
        return dict(kind=kind, dtype="f32", rows=_log_int(rng, 64, 4096),
                    cols=_log_int(rng, 64, 2048), out=_log_int(rng, 64, 2048))
    if kind in ("softmax", "logsumexp"):
        cols = _width(rng, 1000, 151936)
        rows = min(_log_int(rng, 16, 8192), (1 << 28) // cols)
        return dict(kind=kind, dtype=dtype, rows=rows, cols=cols)
    form = rng.choice(["sequence", "token", "position"])
    batch = _log_int(rng, 2, 32)
    rows = _log_int(rng, 32, 2048)
    cols = min(_width(rng, 64, 4096), (1 << 28) // (batch * rows))
    return dict(kind="mul_bcast", dtype=dtype, form=form, batch=batch, rows=rows, cols=cols)


# ---- inputs -------------------------------------------------------------------

class _Gen:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, dtype, std=1.0):
        t = torch.randn(*shape, generator=self.gen, device="cuda")
        return (t.mul_(std) if std != 1.0 else t).to(dtype)

    def gain(self, n, dtype):
        return (torch.rand(n, generator=self.gen, device="cuda") + 0.5).to(dtype)


def _factor_shape(case):
    """The shape of the broadcast factor of a [batch, rows, cols] tensor: a scale per
    sequence and channel, per token, or per position and channel."""
    b, t, d = case["batch"], case["rows"], case["cols"]
    return {"sequence": (b, 1, d), "token": (b, t, 1), "position": (t, d)}[case["form"]]


def prepare(case, seed):
    g = _Gen(seed)
    dt = DTYPES[case["dtype"]]
    k, rows, cols = case["kind"], case["rows"], case["cols"]
    s = {"kind": k}
    if k in ("rmsnorm", "rms_mul"):
        s["x"] = g.normal(rows, cols, dtype=dt)
        s["gamma"] = g.gain(cols, dt)
        s["dy"] = g.normal(rows, cols, dtype=dt)
    elif k in ("norm_linear", "norm_linear_infer"):
        out = case["out"]
        s["x"] = g.normal(rows, cols, dtype=dt)
        s["gamma"] = g.gain(cols, dt)
        s["W"] = g.normal(cols, out, dtype=dt, std=0.02)
        if k == "norm_linear":
            s["dy"] = g.normal(rows, out, dtype=dt)
    elif k == "linear":
        out = case["out"]
        s["x"] = g.normal(rows, cols, dtype=dt)
        s["w"] = g.normal(out, cols, dtype=dt, std=0.02)
        s["bias"] = g.normal(out, dtype=dt, std=0.1)
        s["dy"] = g.normal(rows, out, dtype=dt)
    elif k == "matmul_f32":
        out = case["out"]
        s["a"] = g.normal(rows, cols, dtype=dt)
        s["b"] = g.normal(cols, out, dtype=dt, std=0.02)
        s["dy"] = g.normal(rows, out, dtype=dt)
    elif k == "softmax":
        s["z"] = g.normal(rows, cols, dtype=dt, std=3.0)
        s["dy"] = g.normal(rows, cols, dtype=dt)
    elif k == "logsumexp":
        s["z"] = g.normal(rows, cols, dtype=dt, std=3.0)
        s["dy"] = g.normal(rows, 1, dtype=dt)
    elif k == "layernorm":
        s["x"] = g.normal(rows, cols, dtype=dt).add_(0.25)
        s["dy"] = g.normal(rows, cols, dtype=dt)
    else:
        shape = (case["batch"], rows, cols)
        s["a"] = g.normal(*shape, dtype=dt)
        s["b"] = g.normal(*_factor_shape(case), dtype=dt)
        s["dy"] = g.normal(*shape, dtype=dt)
    return s


# ---- one pass -------------------------------------------------------------------

def run(s):
    k = s["kind"]
    if k == "rmsnorm":
        y, inv = agk.rmsnorm_fwd(s["x"], s["gamma"], EPS)
        dx, dgamma = agk.rmsnorm_bwd(s["x"], s["gamma"], inv, s["dy"])
        return {"y": y, "inv_rms": inv, "dx": dx, "dgamma": dgamma}
    if k == "rms_mul":
        r, inv = agk.rmsnorm_fwd(s["x"], None, EPS)
        y = agk.mul_rowbcast_fwd(r, s["gamma"])
        dr, dx, dgamma = agk.rms_mul_bwd(s["x"], s["gamma"], inv, s["dy"])
        return {"y": y, "dr": dr, "dx": dx, "dgamma": dgamma}
    if k == "norm_linear":
        y, h, inv = agk.rmsnorm_linear_fwd(s["x"], s["gamma"], s["W"], EPS)
        dx, dgamma, dW = agk.rmsnorm_linear_bwd(s["x"], s["gamma"], inv, h, s["W"], s["dy"])
        return {"y": y, "dx": dx, "dgamma": dgamma, "dW": dW}
    if k == "norm_linear_infer":
        return {"y": agk.rmsnorm_linear_fwd(s["x"], s["gamma"], s["W"], EPS)[0]}
    if k == "linear":
        y = agk.linear_bf16(s["x"], s["w"], s["bias"])
        dw = agk.gemm_bf16(s["dy"], s["x"], trans_a=True, out_dtype=torch.float32)
        db = agk.sum_rows(s["dy"])
        dx = agk.gemm_bf16(s["dy"], s["w"])
        return {"y": y, "dx": dx, "dw": dw, "db": db}
    if k == "matmul_f32":
        y = agk.gemm_f32(s["a"], s["b"])
        da = agk.gemm_f32(s["dy"], s["b"], trans_b=True)
        db = agk.gemm_f32(s["a"], s["dy"], trans_a=True)
        return {"y": y, "da": da, "db": db}
    if k == "softmax":
        y = agk.softmax_fwd(s["z"])
        return {"y": y, "dz": agk.softmax_bwd(y, s["dy"])}
    if k == "logsumexp":
        y, lse = agk.logsumexp_fwd_keep(s["z"])
        return {"y": y, "lse": lse, "dz": agk.logsumexp_bwd_from_value(s["z"], lse, s["dy"])}
    if k == "layernorm":
        y, mean, rstd = agk.layernorm_fwd(s["x"], 1e-5)
        return {"y": y, "mean": mean, "rstd": rstd,
                "dx": agk.layernorm_bwd(s["x"], mean, rstd, s["dy"])}
    y = agk.mul_bcast_fwd(s["a"], s["b"])
    da, db = agk.mul_bcast_bwd(s["dy"], s["a"], s["b"])
    return {"y": y, "da": da, "db": db}


# ---- what a pass cannot do without -----------------------------------------------

def work(case):
    k, rows, cols = case["kind"], case["rows"], case["cols"]
    es = 4 if case["dtype"] == "f32" else 2
    n = rows * cols
    if k == "rmsnorm":    # x in both directions (dy exists only after the forward), dy, y, dx
        return {"bytes": 5 * n * es + 2 * cols * es + 8 * rows + 4 * cols, "flops": 12 * n}
    if k == "rms_mul":    # as rmsnorm, plus dr, the gradient of the inner node
        return {"bytes": 6 * n * es + 3 * cols * es + 8 * rows + 4 * cols, "flops": 13 * n}
    if k == "norm_linear":
        out = case["out"]
        return {"bytes": es * (3 * n + 2 * cols * out + 2 * rows * out) + 4 * cols * out
                + (2 * es + 4) * cols, "flops": 6 * n * out}
    if k == "norm_linear_infer":
        out = case["out"]
        return {"bytes": es * (n + cols + cols * out + rows * out), "flops": 2 * n * out}
    if k == "linear":
        out = case["out"]
        return {"bytes": es * (3 * n + 2 * cols * out + 2 * rows * out + out)
                + 4 * (cols * out + out), "flops": 6 * n * out}
    if k == "matmul_f32":
        out = case["out"]
        return {"bytes": 4 * (3 * n + 3 * cols * out + 2 * rows * out), "flops": 6 * n * out}
    if k == "softmax":    # z, dy in; y out and in again; dz out
        return {"bytes": 5 * n * es, "flops": 9 * n}
    if k == "logsumexp":  # z in both directions; dz out
        return {"bytes": 3 * n * es + rows * (2 * es + 8), "flops": 8 * n}
    if k == "layernorm":
        return {"bytes": 5 * n * es + 16 * rows, "flops": 15 * n}
    n *= case["batch"]    # a twice, dy once; y, da out; the factor twice and its gradient
    m = math.prod(_factor_shape(case))
    return {"bytes": 5 * n * es + m * (2 * es + 4), "flops": 4 * n}


# About four times the 2-norm errors measured against exact() on MI355X:
#  - bf16: 1.5e-3 to 2.4e-3 (one or two roundings to bf16; 1.5e-3 to 1.7e-3 where
#    there is one);
#  - fp32 products: 3e-7 to 8e-7 over 64 to 2048 terms, growing with their number;
#  - the other fp32 kinds: at most 3.3e-7 (dgamma's sum over 65536 rows, the
#    log-sum-exp's exponential).
def tolerance(case):
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 4e-6 if case["kind"] == "matmul_f32" else 1.5e-6}


# ---- the same in 64 bits ------------------------------------------------------------

def _norm_vjp(x, gamma, dy):
    """Inverse rms, dx and dgamma of x * rsqrt(mean(x^2) + EPS) * gamma."""
    inv = (x.square().mean(-1, keepdim=True) + EPS).rsqrt()
    xh = x * inv
    dgamma = (dy * xh).sum(0)
    gy = dy * gamma
    dx = (gy - xh * (gy * xh).mean(-1, keepdim=True)) * inv
    return inv, dx, dgamma


def exact(case, seed):
    s = {k: v.double() if torch.is_tensor(v) else v for k, v in prepare(case, seed).items()}
    k = s["kind"]
    if k == "rmsnorm":
        inv, dx, dgamma = _norm_vjp(s["x"], s["gamma"], s["dy"])
        return {"y": s["x"] * inv * s["gamma"], "inv_rms": inv[:, 0], "dx": dx, "dgamma": dgamma}
    if k == "rms_mul":
        inv, dx, dgamma = _norm_vjp(s["x"], s["gamma"], s["dy"])
        return {"y": s["x"] * inv * s["gamma"], "dr": s["dy"] * s["gamma"], "dx": dx,
                "dgamma": dgamma}
    if k in ("norm_linear", "norm_linear_infer"):
        x, gamma, W = s["x"], s["gamma"], s["W"]
        h = x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * gamma
        y = h @ W
        if k == "norm_linear_infer":
            return {"y": y}
        _, dx, dgamma = _norm_vjp(x, gamma, s["dy"] @ W.t())
        return {"y": y, "dx": dx, "dgamma": dgamma, "dW": h.t() @ s["dy"]}
    if k == "linear":
        x, w, dy = s["x"], s["w"], s["dy"]
        return {"y": x @ w.t() + s["bias"], "dx": dy @ w, "dw": dy.t() @ x, "db": dy.sum(0)}
    if k == "matmul_f32":
        return {"y": s["a"] @ s["b"], "da": s["dy"] @ s["b"].t(), "db": s["a"].t() @ s["dy"]}
    if k == "softmax":
        y = torch.softmax(s["z"], -1)
        return {"y": y, "dz": y * (s["dy"] - (y * s["dy"]).sum(-1, keepdim=True))}
    if k == "logsumexp":
        lse = torch.logsumexp(s["z"], -1, keepdim=True)
        return {"y": lse, "lse": lse, "dz": s["dy"] * (s["z"] - lse).exp_()}
    if k == "layernorm":
        x, dy = s["x"], s["dy"]
        mean = x.mean(-1, keepdim=True)
        rstd = ((x - mean).square().mean(-1, keepdim=True) + 1e-5).rsqrt()
        xh = (x - mean) * rstd
        dx = rstd * (dy - dy.mean(-1, keepdim=True) - xh * (dy * xh).mean(-1, keepdim=True))
        return {"y": xh, "mean": mean, "rstd": rstd, "dx": dx}
    a, b, dy = s["a"], s["b"], s["dy"]
    axis = {"sequence": 1, "token": 2, "position": 0}[case["form"]]
    db = (dy * a).sum(axis, keepdim=case["form"] != "position")
    return {"y": a * b, "da": dy * b, "db": db}
