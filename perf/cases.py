"""The work whose speed this repository is held to, as calls of its public entry points.

The framework trains fp32 models: its users call single layers through the C ABI's Python
binding (`ehip.Backend`, on torch CUDA tensors) and whole models through the engine's
resident trainers (`engine_capi.Trainer`). A case is one layer's forward and backward, or
some training steps followed by reading the weights.

  listed()              the cases, each a dict of plain values with a name
  draw(rng)             one more case of the same ranges
  prepare(case, seed)   what the caller holds before the call, on the GPU
  run(state)            one pass; returns its outputs
  work(case)            bytes and operations a pass cannot do without
  tolerance(case)       how far another correct fp32 implementation may be off
  exact(case, seed)     the same outputs in 64 bits from plain torch
"""
import math
import os
import sys

import numpy as np
import torch

# Imported from the repository's root, which is the working folder.
_PACKAGE = os.path.join(os.getcwd(), "cpp-ai-engine_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import ehip  # noqa: E402
import engine_capi  # noqa: E402
import workloads  # noqa: E402

_handles = {}


def backend():
    if "ehip" not in _handles:
        _handles["ehip"] = ehip.Backend()
    return _handles["ehip"]


def engine():
    if "engine" not in _handles:
        _handles["engine"] = engine_capi.Engine()
    return _handles["engine"]


# ----------------------------------------------------------------------- the cases

# Linear(in, out) over `rows` rows: y = x w + b, then dx, dw and db.
LINEAR = [
    # The classifier head of the small CNN (batch 64): two launches of microseconds.
    {"name": "linear_head", "kind": "linear", "rows": 64, "inp": 784, "out": 10},
    # The character model's first feed-forward layer (32 x 64 tokens, d_model 96).
    {"name": "linear_char", "kind": "linear", "rows": 2048, "inp": 96, "out": 384},
    # A layer whose three sizes are odd: every tile has an edge and no row is aligned.
    {"name": "linear_odd", "kind": "linear", "rows": 1999, "inp": 777, "out": 1531},
    # The scaled Transformer's first feed-forward layer (16 x 512 tokens, d_model 1024).
    {"name": "linear_ffn", "kind": "linear", "rows": 8192, "inp": 1024, "out": 4096},
]
# Multi-head attention of projected activations: weights and output, then dq, dk, dv.
ATTENTION = [
    # The character model's (seq 64, heads of 24, causal).
    {"name": "attention_char", "kind": "attention", "batch": 32, "seq": 64, "heads": 4,
     "head_dim": 24, "causal": True},
    # The scaled Transformer's (seq 512, 16 heads of 64, causal).
    {"name": "attention_lm", "kind": "attention", "batch": 16, "seq": 512, "heads": 16,
     "head_dim": 64, "causal": True},
]
ROWS = [
    # The scaled Transformer's LayerNorm, forward and backward.
    {"name": "layernorm_lm", "kind": "layernorm", "rows": 8192, "cols": 1024},
    # A language model's loss over a large vocabulary: mean, probabilities, d logits.
    {"name": "loss_vocab", "kind": "loss", "rows": 8192, "cols": 32000},
]
CONV = [
    # A residual network's middle stage, forward, dx, dw and db.
    {"name": "conv_wide", "kind": "conv", "batch": 32, "cin": 128, "hw": 28, "cout": 128,
     "k": 3, "stride": 1},
]
# Whole training steps (forward, backward, Adam) on a resident batch, then the weights.
STEPS = [
    # The small CNN on 28 x 28 images, batch 64: launch-bound steps.
    {"name": "cnn_steps", "kind": "cnn", "batch": 64, "hw": 28, "c1": 8, "c2": 16, "steps": 10},
    # The character model: d_model 96, 4 heads, two blocks.
    {"name": "char_steps", "kind": "lm", "batch": 32, "seq": 64, "vocab": 121, "d": 96,
     "heads": 4, "ff": 384, "layers": 2, "lr": 1e-3, "steps": 10},
    # Two blocks of the scaled Transformer (d_model 1024, 16 heads, 16 x 512 tokens).
    {"name": "lm_steps", "kind": "lm", "batch": 16, "seq": 512, "vocab": 256, "d": 1024,
     "heads": 16, "ff": 4096, "layers": 2, "lr": 1e-4, "steps": 8},
]


def listed():
    return LINEAR + ATTENTION + ROWS + CONV + STEPS


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "attention", "attention", "layernorm",
                       "loss", "conv", "conv", "cnn", "lm"])
    while True:
        if kind == "linear":
            c = {"rows": _log(rng, 16, 8192), "inp": _log(rng, 16, 4096),
                 "out": _log(rng, 10, 4096)}
            if rng.random() < 0.5:  # widths as models have them: multiples of 16
                c["inp"], c["out"] = -(-c["inp"] // 16) * 16, -(-c["out"] // 16) * 16
            if c["rows"] * c["inp"] * c["out"] > 8192 * 1024 * 4096:
                continue
        elif kind == "attention":
            c = {"batch": _log(rng, 1, 32), "seq": _log(rng, 16, 512), "heads": rng.randint(1, 16),
                 "head_dim": 8 * rng.randint(1, 16), "causal": rng.random() < 0.7}
            if c["batch"] * c["heads"] * c["seq"] ** 2 * c["head_dim"] > 256 * 512 ** 2 * 64:
                continue
        elif kind == "layernorm":
            c = {"rows": _log(rng, 32, 16384), "cols": _log(rng, 16, 4096)}
            if c["rows"] * c["cols"] > 2 ** 25:
                continue
        elif kind == "loss":
            c = {"rows": _log(rng, 16, 8192), "cols": _log(rng, 10, 32000)}
        elif kind == "conv":
            c = {"batch": _log(rng, 1, 64), "cin": _log(rng, 3, 256), "hw": rng.randint(7, 56),
                 "cout": _log(rng, 16, 256), "k": rng.choice([1, 3, 3, 3, 5]),
                 "stride": rng.choice([1, 1, 2])}
            if (c["batch"] * c["hw"] ** 2 * c["cin"] * c["cout"] * c["k"] ** 2
                    > 2 * 32 * 784 * 128 * 128 * 9):
                continue
        elif kind == "cnn":
            c = {"batch": _log(rng, 8, 256), "hw": 4 * rng.randint(4, 8),
                 "c1": rng.randint(4, 12), "c2": rng.randint(8, 24), "steps": 10}
        else:
            heads, hd = rng.randint(1, 8), 8 * rng.randint(2, 8)
            c = {"batch": _log(rng, 2, 32), "seq": _log(rng, 16, 256), "vocab": _log(rng, 32, 512),
                 "d": heads * hd, "heads": heads, "ff": 4 * heads * hd,
                 "layers": rng.randint(1, 4), "lr": 1e-3, "steps": 6}
        c["kind"] = kind
        return c


# --------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale


def _uniform(g, shape, limit):
    return (torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * 2 - 1) * limit


def _inputs(case, seed):
    """The case's device tensors (layers) or host arrays (trainers), from the seed alone."""
    kind = case["kind"]
    if kind == "linear":
        r, i, o = case["rows"], case["inp"], case["out"]
        g = _gen(seed)
        # Normalised activations, Xavier weights, gradients of a mean loss.
        return {"x": _normal(g, (r, i)), "w": _uniform(g, (i, o), math.sqrt(6.0 / (i + o))),
                "b": _normal(g, (o,), 0.02), "dy": _normal(g, (r, o), 1e-3)}
    if kind == "attention":
        g = _gen(seed)
        shape = (case["batch"], case["seq"], case["heads"] * case["head_dim"])
        t = {n: _normal(g, shape) for n in ("q", "k", "v")}
        t["g"] = _normal(g, shape, 1e-3)
        return t
    if kind == "layernorm":
        g = _gen(seed)
        r, c = case["rows"], case["cols"]
        return {"x": _normal(g, (r, c), 2.0) + 0.5, "gamma": _normal(g, (c,), 0.1) + 1.0,
                "beta": _normal(g, (c,), 0.1), "dy": _normal(g, (r, c), 1e-3)}
    if kind == "loss":
        g = _gen(seed)
        r, c = case["rows"], case["cols"]
        return {"logits": _normal(g, (r, c), 2.0),
                "targets": torch.randint(0, c, (r,), generator=g, device="cuda",
                                         dtype=torch.int32),
                "one": torch.ones(1, device="cuda")}
    if kind == "conv":
        g = _gen(seed)
        n, ci, hw, co, k, s = (case[x] for x in ("batch", "cin", "hw", "cout", "k", "stride"))
        o = (hw + 2 * (k // 2) - k) // s + 1
        return {"x": torch.relu(_normal(g, (n, ci, hw, hw))),
                "w": _uniform(g, (co, ci, k, k), math.sqrt(6.0 / (ci * k * k))),
                "b": _normal(g, (co,), 0.02), "g": _normal(g, (n, co, o, o), 1e-3)}
    if kind == "cnn":
        r = np.random.default_rng(seed)
        n, hw, c1, c2 = case["batch"], case["hw"], case["c1"], case["c2"]
        flat = c2 * (hw // 4) ** 2
        params = []
        for shape, fan in (((c1, 1, 3, 3), 9), ((c1,), 0), ((c2, c1, 3, 3), 9 * c1), ((c2,), 0),
                           ((flat, 10), flat), ((10,), 0)):
            size = int(np.prod(shape))
            lim = math.sqrt(6.0 / fan) if fan else 0.0
            params.append(r.uniform(-lim, lim, size).astype(np.float32) if fan
                          else np.zeros(size, np.float32))
        return {"x": r.uniform(0.0, 1.0, (n, 1, hw, hw)).astype(np.float32),
                "labels": r.integers(0, 10, n), "params": np.concatenate(params)}
    ids, targets = workloads.lm_inputs(seed, case["batch"], case["seq"], case["vocab"])
    params = workloads.lm_init_params(seed + 1, case["vocab"], case["d"], case["ff"],
                                      case["layers"])
    return {"ids": ids, "targets": targets, "params": params}


def prepare(case, seed):
    t = _inputs(case, seed)
    state = {"case": case, "t": t}
    if case["kind"] == "cnn":
        state["trainer"] = engine_capi.Trainer.cnn(engine(), t["x"], t["labels"], t["params"],
                                                   lr=1e-3, c1=case["c1"], c2=case["c2"])
    elif case["kind"] == "lm":
        state["trainer"] = engine_capi.Trainer.charlm(
            engine(), t["ids"], t["targets"], case["vocab"], case["d"], case["heads"], case["ff"],
            case["layers"], t["params"], lr=case["lr"])
    else:
        state["hip"] = backend()
    return state


# ------------------------------------------------------------------------------ run

def _product(hip, ta, tb, m, n, k, a, lda, b, ldb, c, ldc, batch=1, inner=1, sa=(0, 0), sb=(0, 0),
             sc=(0, 0), **more):
    d = ehip.GemmEx(trans_a=ta, trans_b=tb, batch=batch, inner=inner, m=m, n=n, k=k,
                    a=a.data_ptr(), lda=lda, stride_a=sa[0], stride_a_inner=sa[1],
                    b=b.data_ptr(), ldb=ldb, stride_b=sb[0], stride_b_inner=sb[1],
                    c=c.data_ptr(), ldc=ldc, stride_c=sc[0], stride_c_inner=sc[1],
                    alpha=1.0, addend_period=1)
    for name, value in more.items():
        setattr(d, name, value)
    hip.gemm_ex(d)
    return c


def _run_linear(hip, c, t):
    r, i, o = c["rows"], c["inp"], c["out"]
    y = _product(hip, 0, 0, r, o, i, t["x"], i, t["w"], o, hip.f32((r, o)), o,
                 addend=t["b"].data_ptr())
    dx, dw, db = hip.linear_backward(t["x"], t["w"], t["dy"])
    return {"y": y, "dx": dx, "dw": dw, "db": db}


def _run_attention(hip, c, t):
    """The engine's attention node: one launch per direction where the sequence and the head
    are short, otherwise the head products and the row softmax between them."""
    n, s, h, hd, causal = c["batch"], c["seq"], c["heads"], c["head_dim"], c["causal"]
    q, k, v, g, d = t["q"], t["k"], t["v"], t["g"], h * hd
    scale = 1.0 / math.sqrt(hd)
    if hip.lib.ehip_attention_short_supported(s, hd):
        w, out = hip.attention_short(q, k, v, h, scale, causal)
        dq, dk, dv = hip.attention_short_backward(q, k, v, w, g, h, scale, causal)
        return {"weights": w, "out": out, "dq": dq, "dk": dk, "dv": dv}
    act, sq = (s * d, hd), (h * s * s, s * s)
    z = dict(batch=n * h, inner=h)
    scores, w = hip.f32((n, h, s, s)), hip.f32((n, h, s, s))
    _product(hip, 0, 1, s, s, hd, q, d, k, d, scores, s, sa=act, sb=act, sc=sq, alpha=scale,
             causal=4 if causal else 0, **z)
    soft = hip.lib.ehip_softmax_causal_f32 if causal else hip.lib.ehip_softmax_f32
    hip.ok(soft(hip.p(scores), hip.p(w), n * h * s, s, hip.stream()), "softmax")
    out = _product(hip, 0, 0, s, hd, s, w, s, v, d, hip.f32((n, s, d)), d, sa=sq, sb=act, sc=act,
                   causal=2 if causal else 0, **z)
    dv = _product(hip, 1, 0, s, hd, s, w, s, g, d, hip.f32((n, s, d)), d, sa=sq, sb=act, sc=act,
                  causal=3 if causal else 0, **z)
    ds = _product(hip, 0, 1, s, s, hd, g, d, v, d, scores, s, sa=act, sb=act, sc=sq,
                  causal=4 if causal else 0, **z)
    back = (hip.lib.ehip_softmax_backward_scaled_causal_f32 if causal
            else hip.lib.ehip_softmax_backward_scaled_f32)
    hip.ok(back(hip.p(w), hip.p(ds), hip.p(ds), n * h * s, s, scale, hip.stream()),
           "softmax backward")
    dq = _product(hip, 0, 0, s, hd, s, ds, s, k, d, hip.f32((n, s, d)), d, sa=sq, sb=act, sc=act,
                  causal=2 if causal else 0, **z)
    dk = _product(hip, 1, 0, s, hd, s, ds, s, q, d, hip.f32((n, s, d)), d, sa=sq, sb=act, sc=act,
                  causal=3 if causal else 0, **z)
    return {"weights": w, "out": out, "dq": dq, "dk": dk, "dv": dv}


def _run_layernorm(hip, c, t):
    out, xhat, inv = hip.layernorm(t["x"], t["gamma"], t["beta"])
    dx, dgamma, dbeta = hip.layernorm_backward(t["dy"], xhat, t["gamma"], inv)
    return {"out": out, "xhat": xhat, "inv_std": inv, "dx": dx, "dgamma": dgamma, "dbeta": dbeta}


def _run_loss(hip, c, t):
    loss, probs = hip.cross_entropy(t["logits"], t["targets"])
    dlogits = hip.cross_entropy_backward(probs, t["targets"], t["one"])
    return {"loss": loss, "probs": probs, "dlogits": dlogits}


def _run_conv(hip, c, t):
    """The engine's Conv2d: direct kernels for narrow layers, implicit GEMM for the others."""
    x, w, b, g, s, p = t["x"], t["w"], t["b"], t["g"], c["stride"], c["k"] // 2
    win = ehip.window(*x.shape, c["k"], c["k"], s, p)
    if hip.lib.ehip_conv2d_direct_supported(win, c["cout"]):
        y = hip.conv2d(x, w, b, s, p)
        dx = hip.conv2d_backward_input(g, w, tuple(x.shape), s, p)
        dw, db = hip.conv2d_backward_weight(x, g, tuple(w.shape), s, p)
    else:
        y = hip.conv2d_igemm(x, w, b, s, p)
        dx, dw, db = hip.conv2d_igemm_backward(x, w, g, s, p)
    return {"y": y, "dx": dx, "dw": dw, "db": db}


_RUN = {"linear": _run_linear, "attention": _run_attention, "layernorm": _run_layernorm,
        "loss": _run_loss, "conv": _run_conv}


def run(state):
    case = state["case"]
    if case["kind"] in _RUN:
        return _RUN[case["kind"]](state["hip"], case, state["t"])
    trainer = state["trainer"]
    for _ in range(case["steps"]):
        trainer.step()
    return {"loss": trainer.loss(), "params": trainer.params()}


# -------------------------------------------------------------- work and tolerances

def work(case):
    kind = case["kind"]
    if kind == "linear":
        r, i, o = case["rows"], case["inp"], case["out"]
        return {"bytes": 8 * (r * i + i * o + r * o + o), "flops": 6 * r * i * o}
    if kind == "attention":
        n, s, h, hd = case["batch"], case["seq"], case["heads"], case["head_dim"]
        pairs = n * h * (s * (s + 1) // 2 if case["causal"] else s * s)
        return {"bytes": 32 * n * s * h * hd + 4 * n * h * s * s, "flops": 12 * pairs * hd}
    if kind == "layernorm":
        n = case["rows"] * case["cols"]
        return {"bytes": 20 * n, "flops": 16 * n}
    if kind == "loss":
        n = case["rows"] * case["cols"]
        return {"bytes": 12 * n, "flops": 6 * n}
    if kind == "conv":
        n, ci, hw, co, k, s = (case[x] for x in ("batch", "cin", "hw", "cout", "k", "stride"))
        o = (hw + 2 * (k // 2) - k) // s + 1
        return {"bytes": 8 * (n * ci * hw * hw + n * co * o * o + co * ci * k * k + co),
                "flops": 6 * n * o * o * co * ci * k * k}
    if kind == "cnn":
        n, hw, c1, c2 = case["batch"], case["hw"], case["c1"], case["c2"]
        macs = n * (hw * hw * c1 * 9 + (hw // 2) ** 2 * c2 * c1 * 9 + c2 * (hw // 4) ** 2 * 10)
        params = 10 * c1 + (9 * c1 + 1) * c2 + c2 * (hw // 4) ** 2 * 10 + 10
        acts = n * (hw * hw + c1 * (hw // 2) ** 2 + c2 * (hw // 4) ** 2)
        return {"bytes": case["steps"] * (8 * acts + 28 * params), "flops": case["steps"] * 6 * macs}
    t, d, ff, v, s = case["batch"] * case["seq"], case["d"], case["ff"], case["vocab"], case["seq"]
    layer = 4 * d * d + 2 * d * ff
    params = case["layers"] * (layer + 9 * d + ff) + 2 * v * d + v
    macs = t * (case["layers"] * (layer + 2 * d * (s + 1) // 2) + d * v)
    acts = t * (case["layers"] * (10 * d + ff) + 2 * d + 2 * v)
    return {"bytes": case["steps"] * (8 * acts + 28 * params), "flops": case["steps"] * 6 * macs}


def tolerance(case):
    """About four times what the kernels' sums differ from 64-bit results by (relative error
    1.1e-6 at K = 8192, 5.6e-7 for the attention gradients, under 2e-7 for the row kernels)."""
    kind = case["kind"]
    if kind in ("linear", "conv"):
        return {"rel": 5e-6, "max": 1e-4}
    if kind == "attention":
        return {"rel": 3e-6, "max": 1e-3}
    if kind in ("layernorm", "loss"):
        return {"rel": 1e-6, "max": 1e-3}
    # Adam divides a gradient by its own size: where the gradient is rounding noise (the key
    # projections' biases) its sign alone moves the weight by lr a step.
    return {"rel": 5e-3, "max": 0.5}


# -------------------------------------------------------------------------- exact

def _heads(x, h):
    n, s, d = x.shape
    return x.reshape(n, s, h, d // h).transpose(1, 2)


def _merge(x):
    n, h, s, hd = x.shape
    return x.transpose(1, 2).reshape(n, s, h * hd)


def _attend(q, k, v, h, causal):
    """(weights, merged output) in the operands' precision."""
    q, k, v = _heads(q, h), _heads(k, h), _heads(v, h)
    s = q.shape[2]
    scores = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(q.shape[3])
    if causal:
        above = torch.ones(s, s, dtype=torch.bool, device=q.device).triu(1)
        scores = scores.masked_fill(above, -math.inf)
    w = torch.softmax(scores, -1)
    return w, _merge(torch.matmul(w, v))


def _conv(x, w, b, stride, pad):
    """Convolution as a product with unfolded columns."""
    n, _, hw, _ = x.shape
    co, _, k, _ = w.shape
    o = (hw + 2 * pad - k) // stride + 1
    cols = torch.nn.functional.unfold(x, k, padding=pad, stride=stride)
    return (torch.matmul(w.reshape(co, -1), cols) + b[:, None]).reshape(n, co, o, o)


def _layer_norm(x, gamma, beta, eps=1e-5):
    mean = x.mean(-1, keepdim=True)
    inv = 1.0 / torch.sqrt(((x - mean) ** 2).mean(-1, keepdim=True) + eps)
    xhat = (x - mean) * inv
    return xhat * gamma + beta, xhat, inv


def _adam_steps(params, loss_of, steps, lr, eps=1e-8):
    """`steps` Adam steps in 64 bits over the flat leaf tensors; (last loss, parameters)."""
    f = lambda v: float(np.float32(v))  # noqa: E731  (the engine takes its constants in fp32)
    b1, b2 = f(0.9), f(0.999)
    m = [torch.zeros_like(p) for p in params]
    v = [torch.zeros_like(p) for p in params]
    loss = None
    for t in range(1, steps + 1):
        leaves = [p.detach().requires_grad_(True) for p in params]
        loss = loss_of(leaves)
        grads = torch.autograd.grad(loss, leaves)
        for i, g in enumerate(grads):
            m[i] = b1 * m[i] + (1 - b1) * g
            v[i] = b2 * v[i] + (1 - b2) * g * g
            params[i] = leaves[i].detach() - f(lr) * (m[i] / (1 - b1 ** t)) / (
                torch.sqrt(v[i] / (1 - b2 ** t)) + f(eps))
    return float(loss.detach()), torch.cat([p.reshape(-1) for p in params]).cpu().numpy()


def _split(flat, shapes):
    out, at = [], 0
    for shape in shapes:
        size = int(np.prod(shape))
        out.append(torch.from_numpy(flat[at:at + size].reshape(shape)).cuda().double())
        at += size
    return out


def exact(case, seed):
    kind, t = case["kind"], _inputs(case, seed)
    if kind == "linear":
        x, w, b, dy = (t[n].double() for n in ("x", "w", "b", "dy"))
        return {"y": x @ w + b, "dx": dy @ w.t(), "dw": x.t() @ dy, "db": dy.sum(0)}
    if kind == "attention":
        q, k, v = (t[n].double().requires_grad_(True) for n in ("q", "k", "v"))
        w, out = _attend(q, k, v, case["heads"], case["causal"])
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), t["g"].double())
        return {"weights": w.detach(), "out": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    if kind == "layernorm":
        x, gamma, beta = (t[n].double().requires_grad_(True) for n in ("x", "gamma", "beta"))
        out, xhat, inv = _layer_norm(x, gamma, beta)
        dx, dg, db = torch.autograd.grad(out, (x, gamma, beta), t["dy"].double())
        return {"out": out.detach(), "xhat": xhat.detach(), "inv_std": inv.detach().reshape(-1),
                "dx": dx, "dgamma": dg, "dbeta": db}
    if kind == "loss":
        x, rows = t["logits"].double(), torch.arange(case["rows"], device="cuda")
        logp = torch.log_softmax(x, -1)
        loss = -logp[rows, t["targets"].long()].mean()
        probs = logp.exp_()
        dlogits = probs.clone()
        dlogits[rows, t["targets"].long()] -= 1.0
        return {"loss": loss.reshape(1), "probs": probs, "dlogits": dlogits / case["rows"]}
    if kind == "conv":
        x, w, b = (t[n].double().requires_grad_(True) for n in ("x", "w", "b"))
        y = _conv(x, w, b, case["stride"], case["k"] // 2)
        dx, dw, db = torch.autograd.grad(y, (x, w, b), t["g"].double())
        return {"y": y.detach(), "dx": dx, "dw": dw, "db": db}
    if kind == "cnn":
        n, hw, c1, c2 = case["batch"], case["hw"], case["c1"], case["c2"]
        x = torch.from_numpy(t["x"]).cuda().double()
        labels = torch.from_numpy(t["labels"]).cuda()
        flat = c2 * (hw // 4) ** 2

        def pool(y):  # 2 x 2 windows, the first maximum
            m, c, a, _ = y.shape
            y = y.reshape(m, c, a // 2, 2, a // 2, 2).permute(0, 1, 2, 4, 3, 5)
            y = y.reshape(m, c, a // 2, a // 2, 4)
            return torch.gather(y, -1, y.detach().argmax(-1, keepdim=True)).squeeze(-1)

        def loss_of(p):
            y = pool(torch.relu(_conv(x, p[0], p[1], 1, 1)))
            y = pool(torch.relu(_conv(y, p[2], p[3], 1, 1)))
            return torch.nn.functional.cross_entropy(y.reshape(n, flat) @ p[4] + p[5], labels)

        params = _split(t["params"], [(c1, 1, 3, 3), (c1,), (c2, c1, 3, 3), (c2,), (flat, 10),
                                      (10,)])
        loss, params = _adam_steps(params, loss_of, case["steps"], 1e-3)
        return {"loss": loss, "params": params}
    n, s, v, d, h, ff = (case[x] for x in ("batch", "seq", "vocab", "d", "heads", "ff"))
    ids = torch.from_numpy(t["ids"]).cuda().long()
    targets = torch.from_numpy(t["targets"]).cuda()
    # The positional table is an input of the model: built in fp32, as the engine builds it.
    i = np.arange(d)
    power = np.power(np.float32(10000.0), (i // 2 * 2).astype(np.float32) / np.float32(d))
    angle = np.arange(s, dtype=np.float32)[:, None] / power[None, :]
    table = np.where(i % 2 == 0, np.sin(angle), np.cos(angle)).astype(np.float32)
    table = torch.from_numpy(table).cuda().double()

    def loss_of(p):
        p = list(p)
        x = p[0][ids] + table
        for i in range(case["layers"]):
            (g1, b1, g2, b2, wq, bq, wk, bk, wv, bv, wo, bo, w1, c1, w2, c2) = p[1 + 16 * i:
                                                                                 17 + 16 * i]
            a = _layer_norm(x, g1, b1)[0]
            x = x + _attend(a @ wq + bq, a @ wk + bk, a @ wv + bv, h, True)[1] @ wo + bo
            a = _layer_norm(x, g2, b2)[0]
            x = x + torch.relu(a @ w1 + c1) @ w2 + c2
        logits = (x @ p[-2] + p[-1]).reshape(n * s, v)
        return torch.nn.functional.cross_entropy(logits, targets)

    shapes = [shape for _, shape, _ in workloads.lm_param_layout(v, d, ff, case["layers"])]
    loss, params = _adam_steps(_split(t["params"], shapes), loss_of, case["steps"], case["lr"])
    return {"loss": loss, "params": params}
