"""Timed workloads of goneuron_amd: the training steps, the inference pass and
the per-layer operators that a user's program calls, over the range of sizes
they are called with.

A case is a dict of plain values; ``prepare`` builds what a program holds
before the call (a compiled model with its weights, inputs on the GPU, an
operator's buffers), ``run`` makes one pass through the public entry points,
``exact`` restates the same pass in float64 torch with the reference's
semantics (per-token Dense gradients from the last token, the loss gradient
fed through the Softmax Jacobian, and so on).

Families (``kind``):
  dense_step   one train step of a Dense stack (forward, backward, Adam)
  predict      one inference pass of a Dense stack
  dense        one Dense layer, forward and backward
  cnn_step     one train step of Conv2D [Conv2D] MaxPool2D Flatten Dense
  conv         one Conv2D layer, forward and backward
  gpt_step     one train step of Embedding, PositionalEncoding,
               TransformerBlock(Ext), CLSPooling, Dense
  mha          one MultiHeadAttention layer, forward and backward
  lstm_step    one train step of SequenceUnroller(LSTM), Dense
  gru          one SequenceUnroller(GRU) layer, forward and backward
  norm         one LayerNorm or RMSNorm layer, forward and backward
"""
import ctypes as C
import math

import numpy as np
import torch
import torch.nn.functional as F

import goneuron_amd as gn
from goneuron_amd import configs
from goneuron_amd._lib import check, lib

LR, BETA1, BETA2, EPS = 1e-3, float(np.float32(0.9)), float(np.float32(0.999)), 1e-8
ACT = {"relu": 1, "sigmoid": 2, "tanh": 3, "linear": 6}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest step a user trains: an MNIST-sized MLP, latency and launches
        dict(name="mlp_step", kind="dense_step", B=64, inp=784, width=128, depth=1, classes=10,
             head="softmax", drop=True),
        # the largest: the wide Dense stack, 71M parameters, matrix products and Adam
        dict(name="wide_step", kind="dense_step", B=1024, inp=4096, width=4096, depth=4, classes=1000,
             head="logsoftmax", drop=False),
        # a layer of sizes nobody rounded: tabular features, a last short batch
        dict(name="dense_ragged", kind="dense", B=333, inp=1001, out=517, act="tanh"),
        # serving the wide stack at a modest batch: every weight read once
        dict(name="predict_wide", kind="predict", B=48, inp=4096, width=4096, depth=4, classes=1000,
             head="logsoftmax"),
        # an image classifier of two convolutions at 32 x 32
        dict(name="cnn_step", kind="cnn_step", B=128, ch=3, hw=32, c1=16, c2=16, classes=10),
        # a convolution deeper in a network, where channels outnumber pixels' colours
        dict(name="conv_mid", kind="conv", B=32, ic=16, hw=32, oc=32, k=3, s=1, p=1, act="linear"),
        # a small language model's step at its usual context
        dict(name="gpt_step", kind="gpt_step", B=32, T=128, vocab=8000, dim=256, heads=8, ff=1024,
             causal=True, act="relu", norm="ln", rope=False),
        # attention over a long context, causal, 64-wide heads
        dict(name="mha_long", kind="mha", B=4, T=512, dim=512, heads=8, causal=True, rope=False),
        # attention over image patches: an odd token count, no mask
        dict(name="mha_patches", kind="mha", B=8, T=197, dim=192, heads=3, causal=False, rope=False),
        # sequence regression with an LSTM
        dict(name="lstm_step", kind="lstm_step", B=64, T=100, inp=64, hidden=256),
        # the same sequences through a GRU layer
        dict(name="gru_seq", kind="gru", B=64, T=100, inp=64, hidden=256),
        # the normalisation of a wider transformer's activations: memory traffic
        dict(name="layernorm", kind="norm", norm="ln", rows=8192, n=1024),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dense_step", "predict", "dense", "cnn_step", "conv", "gpt_step", "mha", "lstm_step",
                       "gru", "norm"])
    if kind == "dense_step":
        return dict(kind=kind, B=_logint(rng, 16, 1024), inp=_logint(rng, 16, 4096), width=_logint(rng, 32, 2048),
                    depth=rng.randint(1, 4), classes=_logint(rng, 2, 1000),
                    head=rng.choice(["softmax", "logsoftmax"]), drop=rng.random() < 0.3)
    if kind == "predict":
        return dict(kind=kind, B=_logint(rng, 1, 1024), inp=_logint(rng, 16, 4096), width=_logint(rng, 32, 4096),
                    depth=rng.randint(1, 4), classes=_logint(rng, 2, 1000),
                    head=rng.choice(["softmax", "logsoftmax"]))
    if kind == "dense":
        return dict(kind=kind, B=_logint(rng, 1, 4096), inp=_logint(rng, 8, 4096), out=_logint(rng, 8, 4096),
                    act=rng.choice(["linear", "tanh", "sigmoid"]))
    if kind == "cnn_step":
        return dict(kind=kind, B=_logint(rng, 16, 256), ch=rng.choice([1, 3]), hw=rng.randint(12, 48),
                    c1=rng.choice([8, 12, 16, 24]), c2=rng.choice([0, 8, 16, 20]), classes=_logint(rng, 2, 100))
    if kind == "conv":
        while True:
            k = rng.choice([1, 3, 3, 5])
            c = dict(kind=kind, B=_logint(rng, 4, 128), ic=_logint(rng, 1, 64), hw=_logint(rng, 7, 64),
                     oc=_logint(rng, 4, 128), k=k, s=rng.choice([1, 1, 2]), p=rng.randint(0, k // 2),
                     act=rng.choice(["linear", "tanh", "sigmoid"]))
            o = _conv_out(c)
            # the backward's partial weight gradients are bounded by the context's scratch
            if c["B"] * o * c["oc"] * (c["ic"] * k * k + 1) <= 16e6 and 2 * work(c)["flops"] <= 60e9:
                return c
    if kind == "gpt_step":
        heads = rng.choice([2, 4, 8])
        hd = rng.choice([16, 32, 48, 64])
        return dict(kind=kind, B=_logint(rng, 4, 32), T=_logint(rng, 16, 256), vocab=_logint(rng, 100, 8000),
                    dim=heads * hd, heads=heads, ff=heads * hd * rng.choice([2, 4]), causal=rng.random() < 0.6,
                    act=rng.choice(["relu", "gelu", "swiglu"]), norm=rng.choice(["ln", "rms"]),
                    rope=rng.random() < 0.5)
    if kind == "mha":
        while True:
            heads, hd = rng.choice([1, 2, 3, 4, 8, 12]), rng.choice([16, 24, 32, 48, 64, 80, 128])
            c = dict(kind=kind, B=_logint(rng, 1, 32), T=_logint(rng, 16, 1024), dim=heads * hd, heads=heads,
                     causal=rng.random() < 0.5, rope=rng.random() < 0.4)
            if work(c)["flops"] <= 100e9 and c["B"] * heads * c["T"] ** 2 <= 50e6:
                return c
    if kind == "lstm_step":
        B = _logint(rng, 8, 96)
        chunk = -(-B // configs.gpu_workers(B))
        return dict(kind=kind, B=B, T=min(_logint(rng, 10, 120), max(4, 1800 // chunk)), inp=_logint(rng, 4, 128),
                    hidden=rng.choice([24, 48, 64, 96, 128, 160, 200, 256, 320]))
    if kind == "gru":
        return dict(kind=kind, B=_logint(rng, 8, 128), T=_logint(rng, 10, 100), inp=_logint(rng, 4, 128),
                    hidden=rng.choice([20, 48, 64, 100, 128, 160, 192, 256, 320]))
    return dict(kind="norm", norm=rng.choice(["ln", "rms"]), rows=_logint(rng, 64, 32768), n=_logint(rng, 32, 2048))


# ------------------------------------------------------------------ shared pieces
def _conv_out(c):
    return (c["hw"] + 2 * c["p"] - c["k"]) // c["s"] + 1


def _dense_sizes(c):
    return [(c["inp"] if i == 0 else c["width"], c["width"]) for i in range(c["depth"])] + [(c["width"], c["classes"])]


def _gpt_cfg(c):
    g = configs.gpt(B=c["B"], T=c["T"], vocab=c["vocab"], dim=c["dim"], heads=c["heads"], ff=c["ff"],
                    causal=c["causal"], act=c["act"], norm=c["norm"], rope=c["rope"])
    return g


def _gpt_tensors(c):
    """(name, shape) of every parameter in arena order."""
    D, FF, V, T = c["dim"], c["ff"], c["vocab"], c["T"]
    t = [("E", (V, D)), ("PE", (T, D))]
    for n in ("q", "k", "v", "o"):
        t += [("W" + n, (D, D)), ("b" + n, (D,))]
    for n in ("1", "2"):
        t += [("g" + n, (D,))] + ([("e" + n, (D,))] if c["norm"] == "ln" else [])
    t += [("Wa", (FF, D)), ("Va", (FF, D))] if c["act"] == "swiglu" else [("Wa", (FF, D)), ("ba", (FF,))]
    return t + [("Wb", (D, FF)), ("bb", (D,)), ("Wh", (V, D)), ("bh", (V,))]


def _split(flat, tensors):
    got, at = {}, 0
    for name, shape in tensors:
        n = int(np.prod(shape))
        got[name] = flat[at:at + n].view(shape)
        at += n
    return got


def _data(c, seed):
    """The case's inputs and weights, float32 on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1000003 + 17)

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * scale

    def onehot(B, n):
        y = torch.zeros(B, n, device="cuda")
        y[torch.arange(B, device="cuda"), torch.randint(0, n, (B,), generator=g, device="cuda")] = 1.0
        return y

    def dense_params(sizes, gain=2.0):
        p = []
        for j, (i, o) in enumerate(sizes):
            p += [normal(o * i, scale=math.sqrt((gain if j + 1 < len(sizes) else 1.0) / i)), normal(o, scale=0.05)]
        return torch.cat(p)

    k, d = c["kind"], {}
    if k in ("dense_step", "predict"):
        d["x"] = torch.rand(c["B"], c["inp"], generator=g, device="cuda") if c["classes"] == 10 else normal(c["B"], c["inp"])
        d["params"] = dense_params(_dense_sizes(c))
        d["y"] = onehot(c["B"], c["classes"])
    elif k == "dense":
        d["x"], d["gout"] = normal(c["B"], c["inp"]), normal(c["B"], c["out"])
        d["W"], d["b"] = normal(c["out"], c["inp"], scale=1 / math.sqrt(c["inp"])), normal(c["out"], scale=0.05)
    elif k == "cnn_step":
        n, at = c["ch"], []
        for o in [c["c1"]] + ([c["c2"]] if c["c2"] else []):
            at += [normal(o * n * 9, scale=math.sqrt(2 / (9 * n))), normal(o, scale=0.05)]
            n = o
        f = n * (c["hw"] // 2) ** 2
        at += [normal(c["classes"] * f, scale=1 / math.sqrt(f)), normal(c["classes"], scale=0.05)]
        d["params"] = torch.cat(at)
        d["x"], d["y"] = normal(c["B"], c["ch"] * c["hw"] ** 2), onehot(c["B"], c["classes"])
    elif k == "conv":
        o = _conv_out(c)
        n = c["ic"] * c["k"] ** 2
        d["x"], d["gout"] = normal(c["B"], c["ic"], c["hw"], c["hw"]), normal(c["B"], c["oc"], o, o)
        d["params"] = torch.cat([normal(c["oc"] * n, scale=1 / math.sqrt(n)), normal(c["oc"], scale=0.05)])
    elif k == "gpt_step":
        at = []
        for name, shape in _gpt_tensors(c):
            n = int(np.prod(shape))
            if len(shape) == 2:
                at.append(normal(n, scale=0.7 if name == "E" else 1 / math.sqrt(shape[1])))
            else:
                at.append(normal(n, scale=0.1) + (1.0 if name[0] == "g" else 0.0))
        d["params"] = torch.cat(at)
        d["x"] = torch.randint(0, c["vocab"], (c["B"], c["T"]), generator=g, device="cuda").float()
        d["y"] = onehot(c["B"], c["vocab"])
    elif k == "mha":
        D = c["dim"]
        d["x"], d["gout"] = normal(c["B"], c["T"], D), normal(c["B"], c["T"], D)
        d["params"] = torch.cat([t for _ in range(4) for t in (normal(D * D, scale=1 / math.sqrt(D)),
                                                               normal(D, scale=0.05))])
    elif k in ("lstm_step", "gru"):
        I, H, G, R = c["inp"], c["hidden"], 4 if k == "lstm_step" else 3, 4 if k == "lstm_step" else 2
        at = [normal(G * H * I, scale=1.2 / math.sqrt(I + H)), normal(R * H * H, scale=0.8 / math.sqrt(I + H)),
              normal(G * H, scale=0.1)]
        d["x"] = normal(c["B"], c["T"], I)
        if k == "lstm_step":
            at += [normal(H, scale=1 / math.sqrt(H)), normal(1, scale=0.05)]
            d["y"] = normal(c["B"], 1)
        else:
            d["gout"] = normal(c["B"], H, scale=0.01)
        d["params"] = torch.cat(at)
    else:
        d["x"], d["gout"] = normal(c["rows"], c["n"]) * 1.5 + 0.3, normal(c["rows"], c["n"])
        d["gamma"], d["beta"] = normal(c["n"], scale=0.2) + 1.0, normal(c["n"], scale=0.2)
    return d


class _Region:
    """A model's device arena region, for torch.as_tensor (keeps the model alive)."""

    def __init__(self, model, ptr, n):
        self.model = model
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _arena(model):
    p = [C.c_void_p() for _ in range(4)]
    check(model.device.h, lib().gn_model_arena(model.h, *[C.byref(q) for q in p]))
    return [torch.as_tensor(_Region(model, q.value, model.nparams), device="cuda") for q in p]


def _model(c):
    if c["kind"] in ("dense_step", "predict"):
        sizes, ls = _dense_sizes(c), []
        for j, (i, o) in enumerate(sizes[:-1]):
            ls.append(configs.dense(i, o, "relu"))
            if j == 0 and c.get("drop"):
                ls.append({"kind": "dropout", "p": 0.2, "n": o})
        ls.append(configs.dense(*sizes[-1], c["head"], True))
        cfg = dict(num=0, name=c["kind"], B=c["B"], loss="ce", lr=LR, in_len=c["inp"], classes=c["classes"], layers=ls)
    elif c["kind"] == "cnn_step":
        n, ls = c["ch"], []
        for o in [c["c1"]] + ([c["c2"]] if c["c2"] else []):
            ls.append({"kind": "conv2d", "inC": n, "outC": o, "k": 3, "s": 1, "p": 1, "act": "relu"})
            n = o
        f = n * (c["hw"] // 2) ** 2
        ls += [{"kind": "maxpool2d", "k": 2, "s": 2, "p": 0, "inC": n}, {"kind": "flatten", "n": f},
               configs.dense(f, c["classes"], "softmax", True)]
        cfg = dict(num=0, name="cnn", B=c["B"], loss="ce", lr=LR, in_len=c["ch"] * c["hw"] ** 2,
                   classes=c["classes"], layers=ls)
    elif c["kind"] == "gpt_step":
        cfg = _gpt_cfg(c)
    else:
        cfg = configs.lstm(B=c["B"], T=c["T"], inp=c["inp"], hidden=c["hidden"])
    return configs.build(cfg)


def _step_slices(c):
    """Arena slices returned one by one: a Dense stack by layer, a GPT without
    its key projection's weights (their gradient is a sum that vanishes, and
    Adam turns its rounding noise into whole steps), otherwise the whole."""
    if c["kind"] in ("dense_step", "predict"):
        at, out = 0, []
        for i, o in _dense_sizes(c):
            out.append(slice(at, at + i * o + o))
            at += i * o + o
        return out
    if c["kind"] == "gpt_step":
        nd = c["dim"] ** 2 + c["dim"]
        k0 = (c["vocab"] + c["T"]) * c["dim"] + nd
        return [slice(0, k0), slice(k0 + nd, None)]
    return [slice(0, None)]


def prepare(case, seed):
    c, d = case, _data(case, seed)
    k = c["kind"]
    s = {"case": c, "x": d["x"], "dev": gn.GetDefaultDevice()}

    def new(*shape):
        return torch.empty(*shape, device="cuda")

    if k.endswith("_step") or k == "predict":
        m = _model(c)
        p, gr, am, av = _arena(m)
        p.copy_(d["params"])
        s.update(model=m, y=d.get("y"), out=new(c["B"], m.out_size))
        sl = _step_slices(c)
        s["params"], s["grads"] = [p[q] for q in sl], [gr[q] for q in sl]
        s["adam"] = [am, av]
    else:
        s.update({n: d[n] for n in d})
        x = d["x"]
        n = C.c_int64()
        if k == "dense":
            s.update(out=new(c["B"], c["out"]), gW=new(c["out"], c["inp"]), gb=new(c["out"]), gin=torch.empty_like(x),
                     dz=new(c["B"], c["out"]))
        elif k == "conv":
            s.update(out=torch.empty_like(d["gout"]), grads=torch.empty_like(d["params"]), gin=torch.empty_like(x))
        elif k == "mha":
            check(None, lib().gn_mha_workspace(c["B"], c["T"], c["dim"], c["heads"], int(c["rope"]), C.byref(n)))
            s.update(out=torch.empty_like(x), grads=torch.empty_like(d["params"]), gin=torch.empty_like(x),
                     work=new(n.value))
        elif k == "gru":
            check(None, lib().gn_gru_workspace(c["B"], c["T"], c["inp"], c["hidden"], C.byref(n)))
            s.update(out=new(c["B"], c["hidden"]), grads=torch.empty_like(d["params"]), gin=torch.empty_like(x),
                     work=new(n.value))
        else:
            s.update(out=torch.empty_like(x), stats=new(2 * c["rows"]), gin=torch.empty_like(x), gg=new(c["n"]),
                     gbeta=new(c["n"]), work=torch.empty_like(x))
    torch.cuda.synchronize()
    return s


def run(state):
    s, c, L = state, state["case"], lib()
    k, h = c["kind"], state["dev"].h

    def p(name):
        return s[name].data_ptr()

    if k.endswith("_step"):
        check(h, L.gn_model_train_step_device(s["model"].h, p("x"), p("y"), c["B"]))
        return {"grads": s["grads"], "params": s["params"], "adam": s["adam"]}
    if k == "predict":
        check(h, L.gn_model_predict_device(s["model"].h, p("x"), c["B"], p("out")))
        return s["out"]
    if k == "dense":
        a = (c["B"], c["inp"], c["out"], ACT[c["act"]], 0)
        check(h, L.gn_dense_forward(h, p("x"), p("W"), p("b"), p("out"), *a))
        check(h, L.gn_dense_backward(h, p("x"), p("W"), p("out"), p("gout"), p("gW"), p("gb"), p("gin"), p("dz"), *a,
                                     1.0 / c["B"]))
        return {"out": s["out"], "gW": s["gW"], "gb": s["gb"], "gin": s["gin"]}
    if k == "conv":
        a = (c["B"], c["ic"], c["hw"], c["hw"], c["oc"], c["k"], c["s"], c["p"], ACT[c["act"]])
        check(h, L.gn_conv2d_forward(h, p("x"), p("params"), p("out"), *a))
        check(h, L.gn_conv2d_backward(h, p("x"), p("params"), p("out"), p("gout"), p("grads"), p("gin"), *a,
                                      1.0 / c["B"]))
    elif k == "mha":
        a = (c["B"], c["T"], c["dim"], c["heads"], int(c["causal"]), int(c["rope"]))
        check(h, L.gn_mha_forward(h, p("x"), p("params"), p("out"), p("work"), *a))
        check(h, L.gn_mha_backward(h, p("x"), p("params"), p("gout"), p("grads"), p("gin"), p("work"), *a, 1.0 / c["B"]))
    elif k == "gru":
        a = (c["B"], c["T"], c["inp"], c["hidden"])
        check(h, L.gn_gru_seq_forward(h, p("x"), p("params"), p("out"), p("work"), *a, 0))
        check(h, L.gn_gru_seq_backward(h, p("x"), p("params"), p("gout"), p("grads"), p("gin"), p("work"), *a,
                                       1.0 / c["B"], 0))
    elif c["norm"] == "ln":
        a = (c["rows"], c["n"])
        check(h, L.gn_layernorm_forward(h, p("x"), p("gamma"), p("beta"), p("out"), p("stats"), *a, 1e-5))
        check(h, L.gn_layernorm_backward(h, p("gout"), p("x"), p("gamma"), p("stats"), p("gin"), p("gg"), p("gbeta"),
                                         p("work"), *a, 1.0 / c["rows"]))
        return {"out": s["out"], "gin": s["gin"], "gg": s["gg"], "gbeta": s["gbeta"]}
    else:
        a = (c["rows"], c["n"])
        check(h, L.gn_rmsnorm_forward(h, p("x"), p("gamma"), p("out"), p("stats"), *a, 1e-5))
        check(h, L.gn_rmsnorm_backward(h, p("gout"), p("x"), p("gamma"), p("stats"), p("gin"), p("gg"), p("work"), *a,
                                       1.0 / c["rows"]))
        return {"out": s["out"], "gin": s["gin"], "gg": s["gg"]}
    return {"out": s["out"], "grads": s["grads"], "gin": s["gin"]}


# ------------------------------------------------------------------ work and tolerance
def _nparams(c):
    k = c["kind"]
    if k in ("dense_step", "predict"):
        return sum(i * o + o for i, o in _dense_sizes(c))
    if k == "gpt_step":
        return sum(int(np.prod(s)) for _, s in _gpt_tensors(c))
    if k == "cnn_step":
        n, tot = c["ch"], 0
        for o in [c["c1"]] + ([c["c2"]] if c["c2"] else []):
            tot, n = tot + o * n * 9 + o, o
        return tot + c["classes"] * (n * (c["hw"] // 2) ** 2 + 1)
    I, H = c["inp"], c["hidden"]
    return 4 * H * (I + H + 1) + H + 1


def work(case):
    """Floating-point operations and bytes one pass cannot do without: the
    products of the algorithm, each input and weight read once, each result
    written once (a train step also reads and writes weights and moments)."""
    c, k = case, case["kind"]
    if k in ("dense_step", "predict"):
        mm = [2.0 * c["B"] * i * o for i, o in _dense_sizes(c)]
        io = 4.0 * c["B"] * (c["inp"] + c["classes"])
        if k == "predict":
            return {"bytes": 4.0 * _nparams(c) + io, "flops": sum(mm)}
        return {"bytes": 28.0 * _nparams(c) + io, "flops": 3 * sum(mm) - mm[0]}
    if k == "dense":
        return {"bytes": 4.0 * (2 * c["inp"] * c["out"] + 2 * c["B"] * (c["inp"] + c["out"]) + 2 * c["out"]),
                "flops": 6.0 * c["B"] * c["inp"] * c["out"]}
    if k == "cnn_step":
        px = c["B"] * c["hw"] ** 2
        f = [2.0 * 9 * px * c["ch"] * c["c1"]] + ([2.0 * 9 * px * c["c1"] * c["c2"]] if c["c2"] else [])
        n = c["c2"] or c["c1"]
        fc = 2.0 * c["B"] * n * (c["hw"] // 2) ** 2 * c["classes"]
        return {"bytes": 28.0 * _nparams(c) + 4.0 * (px * c["ch"] + c["B"] * c["classes"]),
                "flops": 2 * f[0] + 3 * sum(f[1:]) + 3 * fc}
    if k == "conv":
        o = _conv_out(c)
        return {"bytes": 4.0 * (2 * c["B"] * c["ic"] * c["hw"] ** 2 + 2 * c["B"] * c["oc"] * o * o
                                + 2 * c["oc"] * (c["ic"] * c["k"] ** 2 + 1)),
                "flops": 6.0 * c["B"] * c["oc"] * o * o * c["ic"] * c["k"] ** 2}
    if k == "gpt_step":
        rows, D, FF = c["B"] * c["T"], c["dim"], c["ff"]
        up = 2 if c["act"] == "swiglu" else 1
        lin = 2.0 * rows * (4 * D * D + (1 + up) * D * FF)
        pairs = (0.5 if c["causal"] else 1.0) * c["T"] ** 2
        att = 4.0 * c["B"] * D * pairs
        # input gradients per token; weight gradients from one token per sample
        return {"bytes": 28.0 * _nparams(c) + 4.0 * (rows + c["B"] * c["vocab"]),
                "flops": 2 * lin + lin / c["T"] + 3 * att + 6.0 * c["B"] * D * c["vocab"]}
    if k == "mha":
        rows, D = c["B"] * c["T"], c["dim"]
        pairs = (0.5 if c["causal"] else 1.0) * c["T"] ** 2
        return {"bytes": 4.0 * (4 * rows * D + 8 * (D * D + D)),
                "flops": 2 * 8.0 * rows * D * D + 8.0 * c["B"] * D * D + 12.0 * c["B"] * D * pairs}
    if k == "lstm_step":
        B, T, I, H = c["B"], c["T"], c["inp"], c["hidden"]
        W = configs.gpu_workers(B)
        n = -(-B // W) * T
        gram = W * (n * (n + 1.0)) * (5 * H + I)  # the clipped gradient chains' inner products
        return {"bytes": 28.0 * _nparams(c) + 4.0 * (B * T * I + B),
                "flops": 2.0 * B * T * (H * I + H * H + 8 * H * H) + 8.0 * B * H * I + gram}
    if k == "gru":
        B, T, I, H = c["B"], c["T"], c["inp"], c["hidden"]
        return {"bytes": 4.0 * (2 * B * T * I + 2 * (3 * H * I + 2 * H * H + 3 * H) + 2 * B * H),
                "flops": 2.0 * B * T * (3 * H * I + 3 * H * H) + 2.0 * B * T * (2 * H * H + 2 * H * H + 3 * H * I)}
    return {"bytes": 4.0 * (5 * c["rows"] * c["n"] + 3 * c["n"]), "flops": 20.0 * c["rows"] * c["n"]}


def tolerance(case):
    k = case["kind"]
    if k == "dense_step":
        # a unit whose pre-activation lies within rounding of 0 may take either
        # side of its ReLU: about one in 2 million does, and each moves its
        # layer's gradient by sqrt(1 / units)
        flips = case["B"] * case["width"] * case["depth"] > 20000
        return {"rel": 1e-2 if flips else 2e-5, "max": 0.5}
    if k == "cnn_step":
        return {"rel": 1e-2, "max": 0.5}
    if k in ("gpt_step", "lstm_step"):
        # Adam's first step is the gradient's sign, so weights whose gradient is
        # rounding noise move by a whole step either way
        return {"rel": 6e-5, "max": 0.5}
    return {"rel": 1e-5, "max": 1e-3}


# ------------------------------------------------------------------ the same in float64
def _adam(p, g):
    """Weights and moments after the first Network.Step (timestep + 1 = 2)."""
    eff = LR * math.sqrt(1 - BETA2 ** 2) / (1 - BETA1 ** 2)
    m, v = (1 - BETA1) * g, (1 - BETA2) * g * g
    return p - eff * m / (v.sqrt() + EPS), m, v


def _step_result(c, p, g, known=None):
    q, m, v = _adam(p, g)
    sl = _step_slices(c)
    keep = known or [True] * len(sl)
    return {"grads": [g[i] if k else None for i, k in zip(sl, keep)],
            "params": [q[i] if k else None for i, k in zip(sl, keep)],
            "adam": [m, v] if all(keep) else [None, None]}


def _dropout_mask(n, p):
    seed, u = 42, []
    for _ in range(n):
        seed = (seed * 6364136223846793005 + 1) & (2 ** 64 - 1)
        u.append(np.float32(seed >> 33) / np.float32(2 ** 31))
    return torch.tensor([0.0 if v < np.float32(p) else 1.0 for v in u], dtype=torch.float64, device="cuda")


def _dense_forward(c, P, x):
    h, at = x, 0
    sizes = _dense_sizes(c)
    for j, (i, o) in enumerate(sizes):
        h = h @ P[at:at + i * o].view(o, i).T + P[at + i * o:at + i * o + o]
        at += i * o + o
        if j + 1 < len(sizes):
            h = torch.relu(h)
            if j == 0 and c.get("drop"):
                keep = float(np.float32(1) / (np.float32(1) - np.float32(0.2)))
                h = h * _dropout_mask(o, 0.2) * keep
    return torch.softmax(h, 1) if c["head"] == "softmax" else torch.log_softmax(h, 1)


def _conv(x, w, b, k, s, p):
    """Conv2D of the reference: at k3 s1 p1 the interior rows' first and last
    columns hold the bias alone, with the full convolution's gradient."""
    B, _, H, W = x.shape
    oH, oW = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    z = torch.cat([(w.reshape(w.shape[0], -1) @ F.unfold(q, k, padding=p, stride=s)) for q in x.split(max(1, 4096 * 64 // (oH * oW)))])
    z = z.view(B, -1, oH, oW) + b[:, None, None]
    if (k, s, p) == (3, 1, 1):
        skip = torch.zeros(oH, oW, dtype=torch.bool, device=x.device)
        skip[1:oH - 1, 0] = skip[1:oH - 1, oW - 1] = True
        z = z + torch.where(skip, b[:, None, None] - z, torch.zeros((), dtype=z.dtype, device=z.device)).detach()
    return z


class _TokenDense(torch.autograd.Function):
    """A Dense called once per token: its weight gradient takes every token's
    delta and the last token's input."""

    @staticmethod
    def forward(ctx, x, W, b):
        ctx.save_for_backward(x, W)
        return x @ W.T + b

    @staticmethod
    def backward(ctx, g):
        x, W = ctx.saved_tensors
        s = g.sum(1)
        return g @ W, s.T @ x[:, -1], s.sum(0)


class _TokenAct(torch.autograd.Function):
    """The feed-forward activation of a Dense called per token: the derivative
    is the last token's; GELU values run as identity forward."""

    @staticmethod
    def forward(ctx, z, kind):
        ctx.save_for_backward(z)
        ctx.kind = kind
        return torch.relu(z) if kind == "relu" else z.clone()

    @staticmethod
    def backward(ctx, g):
        z = ctx.saved_tensors[0][:, -1:]
        if ctx.kind == "relu":
            return g * (z > 0).to(g.dtype), None
        k = 0.7978845608028654
        t = torch.tanh(k * (z + 0.044715 * z ** 3))
        return g * (0.5 * (1 + t) + 0.5 * z * (1 - t * t) * k * (1 + 3 * 0.044715 * z ** 2)), None


class _TokenSwiGLU(torch.autograd.Function):
    """SwiGLU called per token: only token 0's backward runs, on the last
    token's input, gate and up projection."""

    @staticmethod
    def forward(ctx, x, Wg, Vu):
        ctx.save_for_backward(x, Wg, Vu)
        a = x @ Wg.T
        return a * torch.sigmoid(a) * (x @ Vu.T)

    @staticmethod
    def backward(ctx, gm):
        x, Wg, Vu = ctx.saved_tensors
        xl = x[:, -1]
        a, u = xl @ Wg.T, xl @ Vu.T
        sig = torch.sigmoid(a)
        du, dg = gm[:, 0] * a * sig, gm[:, 0] * (a * sig + sig * (1 - a * sig)) * u
        dx = torch.zeros_like(x)
        dx[:, 0] = dg @ Wg + du @ Vu
        return dx, dg.T @ xl, du.T @ xl


class _LayerNorm(torch.autograd.Function):
    """The reference's backward divides its last term by N std^2."""

    @staticmethod
    def forward(ctx, x, gam, bet):
        mu = x.mean(-1, keepdim=True)
        std = torch.sqrt(((x - mu) ** 2).mean(-1, keepdim=True) + 1e-5)
        ctx.save_for_backward(x, mu, std, gam)
        return gam * (x - mu) / std + bet

    @staticmethod
    def backward(ctx, g):
        x, mu, std, gam = ctx.saved_tensors
        n, gp, d = x.shape[-1], g * gam, x - mu
        dx = (gp - gp.mean(-1, keepdim=True)) / std - d * (gp * d).sum(-1, keepdim=True) / (n * std * std)
        return dx, (g * d / std).flatten(0, -2).sum(0), g.flatten(0, -2).sum(0)


class _RMSNorm(torch.autograd.Function):
    """The reference's backward scales its projection term by gamma_j too."""

    @staticmethod
    def forward(ctx, x, gam):
        r = torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)
        ctx.save_for_backward(x, r, gam)
        return x / r * gam

    @staticmethod
    def backward(ctx, g):
        x, r, gam = ctx.saved_tensors
        s = (g * gam * x).sum(-1, keepdim=True)
        return gam / r * (g - x * s / (x.shape[-1] * r * r)), (g * x / r).flatten(0, -2).sum(0)


def _rope(z, T, heads, hd):
    half = hd // 2
    th = np.array([np.float32(math.pow(10000.0, -2.0 * i / hd)) for i in range(half)], np.float32)
    m = (np.arange(T, dtype=np.float32)[:, None] * th[None, :]).astype(np.float64)
    cs = torch.tensor(np.cos(m).astype(np.float32).astype(np.float64), device=z.device)[:, None]
    sn = torch.tensor(np.sin(m).astype(np.float32).astype(np.float64), device=z.device)[:, None]
    q = z.view(z.shape[0], T, heads, hd)
    a, b = q[..., :half], q[..., half:2 * half]
    return torch.cat([a * cs - b * sn, a * sn + b * cs, q[..., 2 * half:]], 3).reshape(z.shape)


def _attention(q, k, v, c):
    B, T, D = q.shape
    hd = D // c["heads"]
    if c["rope"]:
        q, k = _rope(q, T, c["heads"], hd), _rope(k, T, c["heads"], hd)
    q, k, v = (z.view(B, T, c["heads"], hd).transpose(1, 2).contiguous() for z in (q, k, v))
    s = q @ k.transpose(2, 3).contiguous() / math.sqrt(hd)
    if c["causal"]:
        s = s.masked_fill(torch.triu(torch.ones(T, T, dtype=torch.bool, device=q.device), 1), -1e9)
    return (torch.softmax(s, 3) @ v).transpose(1, 2).reshape(B, T, D)


def _exact_gpt(c, d):
    P = d["params"].requires_grad_(True)
    t = _split(P, _gpt_tensors(c))
    ids = d["x"].long()
    e = t["E"].detach()[ids].requires_grad_(True)
    h = e + t["PE"]
    q, k, v = (_TokenDense.apply(h, t["W" + n], t["b" + n]) for n in "qkv")
    r1 = h + _TokenDense.apply(_attention(q, k, v, c), t["Wo"], t["bo"])

    def norm(z, n):
        return _LayerNorm.apply(z, t["g" + n], t["e" + n]) if c["norm"] == "ln" else _RMSNorm.apply(z, t["g" + n])

    n1 = norm(r1, "1")
    if c["act"] == "swiglu":
        mid = _TokenSwiGLU.apply(n1, t["Wa"], t["Va"])
    else:
        mid = _TokenAct.apply(_TokenDense.apply(n1, t["Wa"], t["ba"]), c["act"])
    out = norm(n1 + _TokenDense.apply(mid, t["Wb"], t["bb"]), "2")
    lp = torch.log_softmax(out[:, 0] @ t["Wh"].T + t["bh"], 1)
    lp.backward(((lp - d["y"]) / c["B"]).detach())
    g = P.grad.clone()
    # the table's gradient: Embedding.Backward zeroes it first, so each
    # worker's last sample alone contributes
    V, D, B = c["vocab"], c["dim"], c["B"]
    W = configs.gpu_workers(B)
    chunk = -(-B // W)
    gE = torch.zeros(V, D, dtype=torch.float64, device=g.device)
    for b0 in range(0, B, chunk):
        b = min(B, b0 + chunk) - 1
        gE.index_add_(0, ids[b], e.grad[b])
    g[:V * D] = gE.reshape(-1)
    return _step_result(c, P.detach(), g)


def _exact_lstm(c, d):
    """BPTT with the reference's gates (f, g and o read their bias alone), its
    carried dh, the input gradient weights from the last step, and the gradient
    sum of every worker's chain clipped to norm 1 after each step."""
    B, T, I, H = c["B"], c["T"], c["inp"], c["hidden"]
    p, X, y = d["params"], d["x"], d["y"][:, 0]
    Wx, Wh = p[:4 * H * I].view(4 * H, I), p[4 * H * I:4 * H * (I + H)].view(4 * H, H)
    b, at = p[4 * H * (I + H):4 * H * (I + H + 1)], 4 * H * (I + H + 1)
    wd, bd = p[at:at + H], p[at + H]
    f, gg, o = torch.sigmoid(b[H:2 * H]), torch.tanh(b[2 * H:3 * H]), torch.sigmoid(b[3 * H:])
    h = cc = torch.zeros(B, H, dtype=torch.float64, device=p.device)
    hs, cs, ig = [h], [cc], []
    for t in range(T):
        i = torch.sigmoid(b[:H] + X[:, t] @ Wx[:H].T + h @ Wh[:H].T)
        cc = f * cc + i * gg
        h = o * torch.tanh(cc)
        hs.append(h), cs.append(cc), ig.append(i)
    dout = 2 * (h @ wd + bd - y)
    dh, dc = dout[:, None] * wd, torch.zeros_like(h)
    dG = [None] * T
    for t in range(T - 1, -1, -1):
        tc = torch.tanh(cs[t + 1])
        dct = dc + dh * o * (1 - tc * tc)
        dG[t] = torch.cat([dct * gg * ig[t] * (1 - ig[t]), dct * cs[t] * f * (1 - f), dct * ig[t] * (1 - gg * gg),
                           dh * tc * o * (1 - o)], 1)
        dc = dct * f
        dh = dh + dG[t] @ Wh
    dG, hp, xl = torch.stack(dG, 1).flip(1), torch.stack(hs[:T], 1).flip(1), X[:, T - 1]
    gWx, gWh, gb = torch.zeros_like(Wx), torch.zeros_like(Wh), torch.zeros_like(b)
    chunk = -(-B // configs.gpu_workers(B))
    for b0 in range(0, B, chunk):
        b1 = min(B, b0 + chunk)
        D, Q = dG[b0:b1].reshape(-1, 4 * H), hp[b0:b1].reshape(-1, H)
        Z = xl[b0:b1].repeat_interleave(T, 0)
        G = ((D @ D.T) * (Z @ Z.T + Q @ Q.T + 1.0)).cpu().numpy()
        w, nrm = np.zeros(len(G)), 0.0
        for j in range(len(G)):
            n2 = nrm + 2 * float(w[:j] @ G[j, :j]) + G[j, j]
            k = 1.0 / math.sqrt(n2) if n2 > 1 else 1.0
            w[:j] *= k
            w[j] = k
            nrm = k * k * n2
        D = D * torch.tensor(w, device=p.device)[:, None]
        gWx += D.T @ Z
        gWh += D.T @ Q
        gb += D.sum(0)
    g = torch.cat([gWx.reshape(-1), gWh.reshape(-1), gb, dout @ h, dout.sum()[None]]) / B
    return _step_result(c, p, g)


def _exact_gru(c, d):
    """The reference's GRU: the candidate reads the reset gate's recurrent
    block, the backward weights it by 1 - u, has no reset-gate delta, carries
    dh and takes input-weight gradients from the last step's input."""
    B, T, I, H = c["B"], c["T"], c["inp"], c["hidden"]
    p, X = d["params"], d["x"]
    Wx, Wh = p[:3 * H * I].view(3 * H, I), p[3 * H * I:3 * H * I + 2 * H * H].view(2 * H, H)
    b = p[3 * H * I + 2 * H * H:]
    Wu, Wr = Wh[:H], Wh[H:]
    h = torch.zeros(B, H, dtype=torch.float64, device=p.device)
    sv = []
    for t in range(T):
        z = X[:, t] @ Wx.T + b
        u, r = torch.sigmoid(z[:, :H] + h @ Wu.T), torch.sigmoid(z[:, H:2 * H] + h @ Wr.T)
        k = torch.tanh(z[:, 2 * H:] + (r * h) @ Wr.T)
        sv.append((u, r, k, h))
        h = h + u * (k - h)
    out, dh = h, d["gout"]
    gWx, gWh, gb, gin = torch.zeros_like(Wx), torch.zeros_like(Wh), torch.zeros_like(b), torch.zeros_like(X)
    for t in range(T - 1, -1, -1):
        u, r, k, hp = sv[t]
        du, dk = dh * (k - hp) * u * (1 - u), dh * (1 - u) * (1 - k * k)
        dG = torch.cat([du, torch.zeros_like(du), dk], 1)
        gWx += dG.T @ X[:, T - 1]
        gb += dG.sum(0)
        gWh += torch.cat([du.T @ hp, dk.T @ (r * hp)])
        gin[:, t] = dG @ Wx
        dh = dh + du @ Wu + (dk * r) @ Wr + dh * u
    return {"out": out, "grads": torch.cat([gWx.reshape(-1), gWh.reshape(-1), gb]) / B, "gin": gin}


def _dact(out, act):
    return {"linear": torch.ones_like(out), "tanh": 1 - out * out, "sigmoid": out * (1 - out)}[act]


def _act(z, act):
    return {"linear": lambda v: v, "tanh": torch.tanh, "sigmoid": torch.sigmoid}[act](z)


def exact(case, seed):
    c = case
    d = {n: t.double() for n, t in _data(c, seed).items()}
    k, x = c["kind"], d["x"]
    if k == "predict":
        return _dense_forward(c, d["params"], x)
    if k == "dense_step":
        P = d["params"].requires_grad_(True)
        o = _dense_forward(c, P, x)
        o.backward(((o - d["y"]) / c["B"]).detach())
        # where a unit's pre-activation lies within float32 rounding of 0 its
        # gradient has two values: only the output layer's is free of that
        sure = c["B"] * c["width"] * c["depth"] <= 20000
        return _step_result(c, P.detach(), P.grad, [sure] * c["depth"] + [True])
    if k == "dense":
        o = _act(x @ d["W"].T + d["b"], c["act"])
        dz = d["gout"] * _dact(o, c["act"])
        return {"out": o, "gW": dz.T @ x / c["B"], "gb": dz.sum(0) / c["B"], "gin": dz @ d["W"]}
    if k == "cnn_step":
        P = d["params"].requires_grad_(True)
        h, n, at = x.view(c["B"], c["ch"], c["hw"], c["hw"]), c["ch"], 0
        for o in [c["c1"]] + ([c["c2"]] if c["c2"] else []):
            h = torch.relu(_conv(h, P[at:at + o * n * 9].view(o, n, 3, 3), P[at + o * n * 9:at + o * n * 9 + o], 3, 1, 1))
            at, n = at + o * n * 9 + o, o
        h = F.max_pool2d(h, 2, 2).flatten(1)
        f = h.shape[1]
        W, b = P[at:at + c["classes"] * f].view(c["classes"], f), P[at + c["classes"] * f:]
        q = torch.softmax(h @ W.T + b, 1)
        q.backward(((q - d["y"]) / c["B"]).detach())
        return _step_result(c, P.detach(), P.grad)
    if k == "conv":
        P = d["params"].requires_grad_(True)
        x.requires_grad_(True)
        n = c["oc"] * c["ic"] * c["k"] ** 2
        z = _conv(x, P[:n].view(c["oc"], c["ic"], c["k"], c["k"]), P[n:], c["k"], c["s"], c["p"])
        o = _act(z, c["act"]).detach()
        z.backward(d["gout"] * _dact(o, c["act"]))
        return {"out": o, "grads": P.grad / c["B"], "gin": x.grad}
    if k == "gpt_step":
        return _exact_gpt(c, d)
    if k == "mha":
        P = d["params"].requires_grad_(True)
        x.requires_grad_(True)
        D = c["dim"]
        w = [(P[i * (D * D + D):][:D * D].view(D, D), P[i * (D * D + D) + D * D:][:D]) for i in range(4)]
        o = _attention(*(_TokenDense.apply(x, *w[i]) for i in range(3)), c)
        o = _TokenDense.apply(o, *w[3])
        o.backward(d["gout"])
        return {"out": o.detach(), "grads": P.grad / c["B"], "gin": x.grad}
    if k == "lstm_step":
        return _exact_lstm(c, d)
    if k == "gru":
        return _exact_gru(c, d)
    x.requires_grad_(True)
    gam, bet = d["gamma"].requires_grad_(True), d["beta"].requires_grad_(True)
    o = _LayerNorm.apply(x, gam, bet) if c["norm"] == "ln" else _RMSNorm.apply(x, gam)
    o.backward(d["gout"])
    got = {"out": o.detach(), "gin": x.grad, "gg": gam.grad / c["rows"]}
    if c["norm"] == "ln":
        got["gbeta"] = bet.grad / c["rows"]
    return got
