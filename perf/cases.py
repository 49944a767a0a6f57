"""What this framework is timed on: training steps through the tensor engine and the
single layers under them through the C ABI, from the smallest step to the largest product.

A case is a dict of plain values; `op` names the family:

  mlp        a whole training step of Linear -> ReLU -> Linear, softmax cross-entropy, SGD or Adam
  linear     a Linear layer's forward and backward (dx, dW, db)
  matmul     matmul_backward: dA and dB of C = A B
  attention  multi-head attention forward and backward over a packed q | k | v projection
  layernorm  LayerNorm forward and backward
  bias_adam  ReLU + bias backward, then one Adam step, over one weight-sized array
  block      a whole training step of a pre-LN transformer encoder block (MSE, SGD)
  lstm       a whole training step of the two-layer LSTM forecaster (MSE, SGD)

Everything is float32, the only floating type that the framework has.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import numrs_amd as nr
from numrs_amd import nn, optim

# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # The smallest step: a classifier on 28 x 28 images, batch 64.  Launches and host calls.
        {"name": "mlp_step_64", "op": "mlp", "batch": 64, "fin": 784, "hidden": 128,
         "classes": 10, "adam": False, "labels": False},
        # An ordinary step with sizes that no tile divides, integer labels and Adam.
        {"name": "mlp_step_ragged", "op": "mlp", "batch": 1000, "fin": 617, "hidden": 1531,
         "classes": 26, "adam": True, "labels": True},
        # A transformer's first feed-forward projection over 16 x 256 tokens.
        {"name": "linear_ffn", "op": "linear", "tokens": 4096, "fin": 512, "fout": 2048},
        # A layer whose sizes are odd in every dimension.
        {"name": "linear_odd", "op": "linear", "tokens": 1001, "fin": 777, "fout": 1531},
        # The largest: a wide projection over 16384 tokens.
        {"name": "linear_large", "op": "linear", "tokens": 16384, "fin": 1024, "fout": 4096},
        # matmul_backward, the framework's headline.
        {"name": "matmul_backward_2048", "op": "matmul", "M": 2048, "K": 2048, "N": 2048},
        # Attention as the encoder block runs it, and at a long odd sequence.
        {"name": "attention_256", "op": "attention", "batch": 16, "seq": 256, "heads": 8,
         "dh": 64},
        {"name": "attention_odd", "op": "attention", "batch": 4, "seq": 777, "heads": 8,
         "dh": 64},
        # Bandwidth-bound layers.
        {"name": "layernorm_32768", "op": "layernorm", "rows": 32768, "cols": 512},
        {"name": "bias_adam_4096", "op": "bias_adam", "rows": 4096, "cols": 4096},
        # Whole models: an encoder block and a recurrent forecaster.
        {"name": "block_step", "op": "block", "batch": 16, "seq": 256, "heads": 8, "dh": 64,
         "ff": 2048},
        {"name": "lstm_step", "op": "lstm", "batch": 64, "steps": 128, "fin": 64, "hidden": 256},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """A size in [lo, hi], even over its logarithm: half of them multiples of 64 (or powers of
    two below it), as models have them, half whatever comes."""
    n = _log(rng, lo, hi)
    if rng.random() < 0.5:
        n = (n + 32) // 64 * 64 if n >= 64 else 1 << (n.bit_length() - 1)
    return max(lo, min(hi, n))


def draw(rng):
    op = rng.choice(["mlp", "linear", "linear", "matmul", "attention", "layernorm", "bias_adam",
                     "block", "lstm"])
    if op == "mlp":
        return {"op": op, "batch": _size(rng, 16, 4096), "fin": _size(rng, 16, 2048),
                "hidden": _size(rng, 16, 2048), "classes": _size(rng, 2, 1000),
                "adam": rng.random() < 0.5, "labels": rng.random() < 0.5}
    if op == "linear":
        while True:
            t, i, o = _size(rng, 16, 16384), _size(rng, 16, 4096), _size(rng, 16, 4096)
            if t * i * o <= 16384 * 1024 * 4096:
                return {"op": op, "tokens": t, "fin": i, "fout": o}
    if op == "matmul":
        return {"op": op, "M": _size(rng, 16, 4096), "K": _size(rng, 16, 4096),
                "N": _size(rng, 16, 2048)}
    if op == "attention":
        while True:
            b, s, h = _size(rng, 1, 32), _size(rng, 16, 1024), _size(rng, 1, 16)
            if b * h * s * s <= 32 * 1024 * 1024:
                return {"op": op, "batch": b, "seq": s, "heads": h,
                        "dh": rng.choice([32, 40, 64, 64, 80, 128])}
    if op == "layernorm":
        while True:
            r, c = _size(rng, 16, 65536), _size(rng, 16, 4096)
            if r * c <= 1 << 25:
                return {"op": op, "rows": r, "cols": c}
    if op == "bias_adam":
        while True:
            r, c = _size(rng, 16, 8192), _size(rng, 16, 8192)
            if r * c <= 1 << 24:
                return {"op": op, "rows": r, "cols": c}
    if op == "block":
        dh = rng.choice([32, 64, 64])
        heads = rng.randint(2, 8)
        return {"op": op, "batch": _size(rng, 1, 16), "seq": _size(rng, 16, 256), "heads": heads,
                "dh": dh, "ff": _size(rng, 64, 2048)}
    return {"op": "lstm", "batch": _size(rng, 2, 64), "steps": _size(rng, 8, 128),
            "fin": _size(rng, 4, 128), "hidden": rng.choice([64, 100, 128, 256, 256])}


# ---------------------------------------------------------------------------
# What a user's program holds
# ---------------------------------------------------------------------------

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = nr.Context(0)
        nr.set_default_context(_ctx)
    return _ctx


class _Memory:
    """Device memory of the engine as torch sees it (no copy)."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "version": 2,
                                         "strides": None, "data": (int(ptr), False)}


def _view(state, ptr, shape):
    key = (ptr, shape)
    t = state["views"].get(key)
    if t is None:
        t = state["views"][key] = torch.as_tensor(_Memory(ptr, shape), device="cuda")
    return t


def _normal(gen, *shape, scale=1.0):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * scale


def _xavier(rng, fan_out, fan_in):
    a = math.sqrt(6.0 / (fan_in + fan_out))
    return rng.uniform(-a, a, (fan_out, fan_in)).astype(np.float32)


def _inputs(case, seed):
    """The case's inputs, from the seed alone: host arrays for the engine's steps, device
    tensors for the layers."""
    op = case["op"]
    if op in ("mlp", "block", "lstm"):
        rng = np.random.default_rng(seed)
        if op == "mlp":
            B, I, H, C = case["batch"], case["fin"], case["hidden"], case["classes"]
            return {"x": rng.standard_normal((B, I), dtype=np.float32),
                    "w1": _xavier(rng, H, I),
                    "b1": rng.standard_normal(H, dtype=np.float32) * np.float32(0.02),
                    "w2": _xavier(rng, C, H),
                    "b2": rng.standard_normal(C, dtype=np.float32) * np.float32(0.02),
                    "labels": rng.integers(0, C, B).astype(np.int32)}
        if op == "block":
            d, f, n = case["heads"] * case["dh"], case["ff"], case["batch"] * case["seq"]
            return {"w": {"wq": _xavier(rng, d, d), "wk": _xavier(rng, d, d),
                          "wv": _xavier(rng, d, d), "wo": _xavier(rng, d, d),
                          "w1": _xavier(rng, f, d), "w2": _xavier(rng, d, f)},
                    "x": rng.standard_normal((n, d), dtype=np.float32),
                    "t": rng.standard_normal((n, d), dtype=np.float32)}
        B, T, I, H = case["batch"], case["steps"], case["fin"], case["hidden"]
        t = np.arange(T)
        phase = rng.uniform(0.0, 2 * math.pi, (B, I))
        omega = rng.uniform(0.05, 0.5, I)
        x = np.sin(omega[None, None, :] * t[None, :, None] + phase[:, None, :])
        x = (x + rng.normal(0.0, 0.1, x.shape)).astype(np.float32)
        layers = [{"w_ih": _xavier(rng, 4 * H, i), "w_hh": _xavier(rng, 4 * H, H),
                   "b": rng.standard_normal(4 * H, dtype=np.float32) * np.float32(0.02)}
                  for i in (I, H)]
        return {"x": x, "layers": layers, "hw": _xavier(rng, 1, H), "hb": np.zeros(1, np.float32),
                "t": rng.standard_normal((B, 1), dtype=np.float32)}
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if op == "linear":
        T, I, O = case["tokens"], case["fin"], case["fout"]
        return {"x": _normal(gen, T, I), "w": _normal(gen, O, I, scale=1 / math.sqrt(I)),
                "b": _normal(gen, O, scale=0.02), "g": _normal(gen, T, O, scale=1e-3)}
    if op == "matmul":
        M, K, N = case["M"], case["K"], case["N"]
        return {"a": _normal(gen, M, K), "b": _normal(gen, K, N), "g": _normal(gen, M, N)}
    if op == "attention":
        n, d = case["batch"] * case["seq"], case["heads"] * case["dh"]
        return {"qkv": _normal(gen, n, 3 * d), "g": _normal(gen, n, d, scale=1e-2)}
    r, c = case["rows"], case["cols"]
    if op == "layernorm":
        return {"x": _normal(gen, r, c) * 1.5 + 0.25, "gamma": 1 + _normal(gen, c, scale=0.1),
                "beta": _normal(gen, c, scale=0.1), "g": _normal(gen, r, c, scale=1e-2)}
    return {"g": _normal(gen, r, c, scale=1e-2), "z": _normal(gen, r, c),
            "p": _normal(gen, r, c, scale=0.05), "m": _normal(gen, r, c, scale=1e-3),
            "v": _normal(gen, r, c, scale=1e-3).square()}


def _array(ctx, t):
    return nr.DeviceArray(ctx, t.data_ptr(), t.shape, owned=False, base=t)


def _engine_state(state, params):
    state["params"] = params
    state["grads"], state["weights"] = [], []
    for p in params:
        data, grad = p.device_ptrs()
        state["weights"].append(_view(state, data, p.shape()))
        state["grads"].append(_view(state, grad, p.shape()))
    return state


def prepare(case, seed):
    ctx, op, i = _context(), case["op"], _inputs(case, seed)
    s = {"case": case, "ctx": ctx, "views": {}}
    if op == "mlp":
        l1 = nn.Linear.with_weights(case["fin"], case["hidden"], i["w1"], i["b1"])
        l2 = nn.Linear.with_weights(case["hidden"], case["classes"], i["w2"], i["b2"])
        s["model"] = nn.Sequential([l1, nn.ReLU(), l2])
        params = s["model"].parameters()
        s["opt"] = optim.Adam.default(params, 1e-3) if case["adam"] else optim.SGD.simple(params, 0.01)
        s["x"] = nr.Tensor.new(i["x"])
        s["target"] = (i["labels"] if case["labels"] else
                       nr.Tensor.new(np.eye(case["classes"], dtype=np.float32)[i["labels"]]))
        return _engine_state(s, params)
    if op == "block":
        s["model"] = nn.TransformerEncoderBlock(i["w"], case["heads"])
        s["opt"] = optim.SGD.simple(s["model"].parameters(), 1e-3)
        s["x"], s["target"] = nr.Tensor.new(i["x"]), nr.Tensor.new(i["t"])
        return _engine_state(s, s["model"].parameters())
    if op == "lstm":
        s["model"] = nn.LSTMForecaster(i["layers"], i["hw"], i["hb"])
        s["opt"] = optim.SGD.simple(s["model"].parameters(), 1e-3)
        s["x"], s["target"] = nr.Tensor.new(i["x"]), nr.Tensor.new(i["t"])
        return _engine_state(s, s["model"].parameters())
    s.update(i)
    new = lambda *shape: torch.zeros(shape, device="cuda", dtype=torch.float32)  # noqa: E731
    if op == "linear":
        s["y"], s["dx"] = torch.zeros_like(i["g"]), torch.zeros_like(i["x"])
        s["dw"], s["db"] = torch.zeros_like(i["w"]), torch.zeros_like(i["b"])
    elif op == "matmul":
        s["da"], s["db"] = torch.zeros_like(i["a"]), torch.zeros_like(i["b"])
        s["arrays"] = [_array(ctx, s[k]) for k in ("g", "a", "b", "da", "db")]
    elif op == "attention":
        s["out"], s["dqkv"] = torch.zeros_like(i["g"]), torch.zeros_like(i["qkv"])
        s["P"] = new(case["batch"] * case["heads"], case["seq"], case["seq"])
    elif op == "layernorm":
        s["y"], s["dx"] = torch.zeros_like(i["x"]), torch.zeros_like(i["x"])
        s["mean"], s["rstd"] = new(case["rows"]), new(case["rows"])
        s["dgamma"], s["dbeta"] = torch.zeros_like(i["gamma"]), torch.zeros_like(i["beta"])
    else:
        s["dx"], s["db"], s["t"] = torch.zeros_like(i["g"]), new(case["cols"]), 0
        s["arrays"] = {k: _array(ctx, s[k]) for k in ("g", "z", "dx", "db", "p", "m", "v")}
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def _check(ctx, rc):
    if rc != 0:
        raise nr.HipError(rc, nr.load().numrs_hip_last_error(ctx.handle).decode())


def _step(s):
    """One training step: the logits (or predictions), the loss, every gradient and every
    updated parameter, in the engine's own memory."""
    case, model, opt = s["case"], s["model"], s["opt"]
    opt.zero_grad()
    if case["op"] == "block":
        y = model.forward_seq(s["x"], case["batch"], case["seq"])
    else:
        y = model.forward(s["x"])
    if case["op"] != "mlp":
        loss = y.mse_loss(s["target"])
    elif case["labels"]:
        loss = y.cross_entropy_labels(s["target"])
    else:
        loss = y.cross_entropy_loss(s["target"])
    loss.backward()
    opt.step()
    s["live"] = (y, loss)  # their memory stays this state's until its next pass
    return {"y": _view(s, y.device_ptrs()[0], y.shape()),
            "loss": _view(s, loss.device_ptrs()[0], (1,)),
            "grads": s["grads"], "weights": s["weights"]}


def run(s):
    case, ctx, lib = s["case"], s["ctx"], nr.load()
    op, h = case["op"], s["ctx"].handle
    if op in ("mlp", "block", "lstm"):
        return _step(s)
    if op == "linear":
        T, I, O = case["tokens"], case["fin"], case["fout"]
        x, w, b, g = (s[k].data_ptr() for k in ("x", "w", "b", "g"))
        _check(ctx, lib.numrs_hip_linear_forward(h, x, w, b, s["y"].data_ptr(), T, I, O))
        _check(ctx, lib.numrs_hip_linear_backward(
            h, g, x, w, s["dx"].data_ptr(), s["dw"].data_ptr(), s["db"].data_ptr(), T, I, O,
            0, 0, 0, 0))
        return {k: s[k] for k in ("y", "dx", "dw", "db")}
    if op == "matmul":
        g, a, b, da, db = s["arrays"]
        ctx.matmul_backward(g, a, b, da, db)
        return {"da": s["da"], "db": s["db"]}
    if op == "attention":
        B, S, H, D = case["batch"], case["seq"], case["heads"], case["heads"] * case["dh"]
        q, out, dq = s["qkv"].data_ptr(), s["out"].data_ptr(), s["dqkv"].data_ptr()
        k, v, P = q + 4 * D, q + 8 * D, s["P"].data_ptr()
        _check(ctx, lib.numrs_hip_attention_forward_strided(h, q, k, v, 3 * D, P, out, D, B, S, H,
                                                            D))
        _check(ctx, lib.numrs_hip_attention_backward_out_strided(
            h, q, k, v, 3 * D, P, out, s["g"].data_ptr(), D, dq, dq + 4 * D, dq + 8 * D, B, S, H,
            D, 0))
        return {"P": s["P"], "out": s["out"], "dqkv": s["dqkv"]}
    if op == "layernorm":
        r, c = case["rows"], case["cols"]
        x, gamma, beta, g, y, mean, rstd, dx, dgamma, dbeta = (
            s[k].data_ptr() for k in ("x", "gamma", "beta", "g", "y", "mean", "rstd", "dx",
                                      "dgamma", "dbeta"))
        _check(ctx, lib.numrs_hip_layernorm_forward(h, x, gamma, beta, y, mean, rstd, r, c, 1e-5))
        _check(ctx, lib.numrs_hip_layernorm_backward(h, g, x, gamma, mean, rstd, dx, dgamma, dbeta,
                                                     r, c, 0, 0, 0))
        return {k: s[k] for k in ("y", "dx", "dgamma", "dbeta")}
    a = s["arrays"]
    ctx.relu_bias_backward(a["g"], a["z"], a["dx"], a["db"])
    s["t"] += 1
    ctx.adam_step(a["p"], a["dx"], a["m"], a["v"], s["t"])
    return {k: s[k] for k in ("dx", "db", "p", "m", "v")}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    op = case["op"]
    if op == "mlp":
        B, I, H, C = case["batch"], case["fin"], case["hidden"], case["classes"]
        n = I * H + H + H * C + C
        # inputs and logits, each weight and gradient once, weights (and moments) written
        return {"bytes": 4 * (B * I + 2 * B * C + (7 if case["adam"] else 3) * n),
                "flops": 2 * B * (2 * I * H + 3 * H * C)}
    if op == "linear":
        T, I, O = case["tokens"], case["fin"], case["fout"]
        return {"bytes": 4 * (2 * T * I + 2 * T * O + 2 * I * O + 2 * O), "flops": 6 * T * I * O}
    if op == "matmul":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 4 * (2 * M * K + 2 * K * N + M * N), "flops": 4 * M * K * N}
    if op == "attention":
        B, S, H, d = case["batch"], case["seq"], case["heads"], case["dh"]
        return {"bytes": 4 * (8 * B * S * H * d + B * H * S * S), "flops": 12 * B * H * S * S * d}
    if op == "layernorm":
        r, c = case["rows"], case["cols"]
        return {"bytes": 4 * (4 * r * c + 4 * c), "flops": 16 * r * c}
    if op == "bias_adam":
        r, c = case["rows"], case["cols"]
        return {"bytes": 4 * (9 * r * c + c), "flops": 14 * r * c}
    if op == "block":
        d, f = case["heads"] * case["dh"], case["ff"]
        n = case["batch"] * case["seq"]
        p = 4 * d * d + 2 * d * f + 9 * d + f
        return {"bytes": 4 * (3 * n * d + 3 * p),
                "flops": 3 * (2 * n * (4 * d * d + 2 * d * f) + 4 * n * case["seq"] * d)}
    B, T, I, H = case["batch"], case["steps"], case["fin"], case["hidden"]
    p = 4 * H * (I + 3 * H + 2) + H + 1
    return {"bytes": 4 * (B * T * I + 2 * B + 3 * p), "flops": 2 * B * T * 4 * H * (2 * I + 9 * H)}


def tolerance(case):
    """Errors of the float32 sums against float64, times at least four, over the declared sizes:
    products 2.2e-7, attention 5e-7, LayerNorm 2e-7, recurrent steps 1e-6; Adam's first steps
    divide two small numbers, whose float32 bias corrections put 6e-6 into the parameter, and
    where a gradient is near zero its sign, and so one whole step, is rounding."""
    op = case["op"]
    if op in ("linear", "matmul"):
        return {"rel": 4e-6, "max": 4e-5}
    if op in ("attention", "layernorm"):
        return {"rel": 4e-6, "max": 1e-4}
    if op == "bias_adam":
        return {"rel": 2.5e-5, "max": 1e-4}
    return {"rel": 1e-5, "max": 1e-3}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------


def _double(v):
    if isinstance(v, dict):
        return {k: _double(x) for k, x in v.items()}
    if isinstance(v, list):
        return [_double(x) for x in v]
    v = torch.as_tensor(v, device="cuda")
    return v.double() if v.is_floating_point() else v.long()


def _attend(q, k, v, heads, batch, seq):
    d = q.shape[1]
    dh = d // heads
    split = lambda t: t.reshape(batch, seq, heads, dh).permute(0, 2, 1, 3)  # noqa: E731
    q, k, v = split(q), split(k), split(v)
    p = torch.softmax((q @ k.transpose(2, 3).contiguous()) / math.sqrt(dh), -1)
    return p.reshape(batch * heads, seq, seq), (p @ v).permute(0, 2, 1, 3).reshape(batch * seq, d)


def _lstm(x, w_ih, w_hh, b):
    h = c = torch.zeros(x.shape[0], w_hh.shape[1], dtype=x.dtype, device=x.device)
    xs, out = x @ w_ih.T + b, []
    for t in range(x.shape[1]):
        i, f, g, o = (xs[:, t] + h @ w_hh.T).chunk(4, 1)
        c = torch.sigmoid(f) * c + torch.sigmoid(i) * torch.tanh(g)
        h = torch.sigmoid(o) * torch.tanh(c)
        out.append(h)
    return torch.stack(out, 1)


def _step_exact(case, i):
    F = torch.nn.functional
    op = case["op"]
    if op == "mlp":
        params = [i["w1"], i["b1"], i["w2"], i["b2"]]
        for p in params:
            p.requires_grad_()
        y = torch.relu(i["x"] @ params[0].T + params[1]) @ params[2].T + params[3]
        loss = F.cross_entropy(y, i["labels"])
    elif op == "block":
        w, d = i["w"], case["heads"] * case["dh"]
        zeros = lambda n: torch.zeros(n, dtype=torch.float64, device="cuda")  # noqa: E731
        one = lambda: torch.ones(d, dtype=torch.float64, device="cuda")  # noqa: E731
        params = [one(), zeros(d), torch.cat([w["wq"], w["wk"], w["wv"]]), zeros(3 * d), w["wo"],
                  zeros(d), one(), zeros(d), w["w1"], zeros(case["ff"]), w["w2"], zeros(d)]
        for p in params:
            p.requires_grad_()
        g1, c1, wqkv, bqkv, wo, bo, g2, c2, w1, b1, w2, b2 = params
        q, k, v = (F.layer_norm(i["x"], (d,), g1, c1) @ wqkv.T + bqkv).chunk(3, 1)
        a = _attend(q, k, v, case["heads"], case["batch"], case["seq"])[1]
        r = i["x"] + a @ wo.T + bo
        y = r + F.gelu(F.layer_norm(r, (d,), g2, c2) @ w1.T + b1) @ w2.T + b2
        loss = F.mse_loss(y, i["t"])
    else:
        params = [layer[k] for layer in i["layers"] for k in ("w_ih", "w_hh", "b")]
        params += [i["hw"], i["hb"]]
        for p in params:
            p.requires_grad_()
        h = _lstm(_lstm(i["x"], *params[:3]), *params[3:6])
        y = h[:, -1] @ params[6].T + params[7]
        loss = F.mse_loss(y, i["t"])
    grads = list(torch.autograd.grad(loss, params))
    with torch.no_grad():
        if op == "mlp" and case["adam"]:  # the first step: both moments are bias-corrected to g
            weights = [p - 1e-3 * g / (g.abs() + 1e-8) for p, g in zip(params, grads)]
        else:
            lr = 0.01 if op == "mlp" else 1e-3
            weights = [p - lr * g for p, g in zip(params, grads)]
    return {"y": y.detach(), "loss": loss.detach().reshape(1), "grads": grads, "weights": weights}


def exact(case, seed):
    i, op = _double(_inputs(case, seed)), case["op"]
    if op in ("mlp", "block", "lstm"):
        return _step_exact(case, i)
    g = i["g"]
    if op == "linear":
        return {"y": i["x"] @ i["w"].T + i["b"], "dx": g @ i["w"], "dw": g.T @ i["x"],
                "db": g.sum(0)}
    if op == "matmul":
        return {"da": g @ i["b"].T, "db": i["a"].T @ g}
    if op == "attention":
        qkv = i["qkv"].requires_grad_()
        P, out = _attend(*qkv.chunk(3, 1), case["heads"], case["batch"], case["seq"])
        return {"P": P.detach(), "out": out.detach(), "dqkv": torch.autograd.grad(out, qkv, g)[0]}
    if op == "layernorm":
        leaves = [i[k].requires_grad_() for k in ("x", "gamma", "beta")]
        y = torch.nn.functional.layer_norm(leaves[0], (case["cols"],), leaves[1], leaves[2])
        dx, dgamma, dbeta = torch.autograd.grad(y, leaves, g)
        return {"y": y.detach(), "dx": dx, "dgamma": dgamma, "dbeta": dbeta}
    dx = torch.where(i["z"] > 0, g, torch.zeros_like(g))
    m, v = 0.9 * i["m"] + 0.1 * dx, 0.999 * i["v"] + 0.001 * dx * dx
    p = i["p"] - 1e-3 * (m / (1 - 0.9)) / (torch.sqrt(v / (1 - 0.999)) + 1e-8)
    return {"dx": dx, "db": dx.sum(0), "p": p, "m": m, "v": v}
