"""The work this library is measured on, as a program that holds its data in
torch tensors gives it to the package: the configuration programs, a dense
layer's forward and backward products, attention's 16-bit products, the row
regions, an embedding with its gradient, and the standardisation of a
feature matrix.

Every case is a dict of plain values; "kind" names the path and the other
entries its sizes and options. The inputs are drawn on the GPU, wrapped once
as borrowed device tensors (with the views and chains a program keeps), and
results are written to tensors the caller owns.
"""
import math

import numpy as np
import torch

import chelis_amd as C

NP = {"f32": np.float32, "f64": np.float64, "bf16": np.uint16, "f16": np.float16, "i64": np.int64}
TORCH = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16, "f16": torch.float16}
WIDTH = {"f32": 4, "f64": 8, "bf16": 2, "f16": 2}
HEAD = 64        # the transformer block's head width
RATE = 0.1       # the MLP step's dropout and learning rates
LEARN = 0.01
EPS = 1e-5
KEY = 44


def listed():
    return [
        # a least-squares gradient step over a small table: launches and host time
        {"name": "linreg_8192x32_f64", "kind": "linreg", "n": 8192, "d": 32, "dtype": "f64"},
        # one training step of a digit classifier: dropout, cross-entropy, SGD
        {"name": "mlp_1024x784x512x10", "kind": "mlp", "batch": 1024, "d_in": 784, "hidden": 512, "classes": 10},
        # the prefill of one pre-norm transformer block, eight full sequences
        {"name": "block_8x512x1024", "kind": "block", "batch": 8, "seq": 512, "width": 1024},
        # a narrow block over a few short sequences of no round length
        {"name": "block_3x200x512", "kind": "block", "batch": 3, "seq": 200, "width": 512},
        # a dense layer's forward and backward, sizes off every tile
        {"name": "dense_f32_4000x1000x3000", "kind": "dense", "m": 4000, "k": 1000, "n": 3000, "dtype": "f32"},
        # the same in binary64 onto a narrow output (many samples, few outputs)
        {"name": "dense_f64_8192x4096x64", "kind": "dense", "m": 8192, "k": 4096, "n": 64, "dtype": "f64"},
        # attention's score and value products in bf16, a batch of heads
        {"name": "heads_bf16_8x16x512", "kind": "heads", "batch": 8, "heads": 16, "seq": 512, "dh": 64,
         "dtype": "bf16"},
        # softmax and its adjoint: attention-sized rows
        {"name": "softmax_f32_16384x1024", "kind": "softmax", "rows": 16384, "n": 1024, "dtype": "f32"},
        # softmax and its adjoint over a vocabulary of no round size
        {"name": "softmax_f32_1000x32003", "kind": "softmax", "rows": 1000, "n": 32003, "dtype": "f32"},
        # layer norm over rows that are no power of two
        {"name": "layernorm_f32_20000x1000", "kind": "layernorm", "rows": 20000, "n": 1000, "dtype": "f32"},
        # embedding lookup and its gradient, word-like (skewed) ids
        {"name": "embed_8192_of_50000x512", "kind": "embed", "tokens": 8192, "vocab": 50000, "width": 512},
        # column statistics of a sample matrix and the standardised matrix
        {"name": "standardise_16384x4096", "kind": "standardise", "n": 16384, "d": 4096, "dtype": "f32"},
    ]


def _size(rng, lo, hi, step=8):
    """A size in [lo, hi], spread over its logarithm; half of them whole
    multiples of `step`, the others as they fall."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))
    if rng.random() < 0.5:
        v = (v + step // 2) // step * step
    return max(lo, min(hi, v))


def _drawn(rng):
    kind = rng.choice(["linreg", "mlp", "block", "block", "dense", "dense", "heads", "softmax", "softmax", "layernorm",
                       "embed", "standardise"])
    if kind == "linreg":
        return {"kind": kind, "n": _size(rng, 500, 100000), "d": _size(rng, 4, 48), "dtype": "f64"}
    if kind == "mlp":
        return {"kind": kind, "batch": _size(rng, 64, 4096, 64), "d_in": _size(rng, 64, 1024, 16),
                "hidden": _size(rng, 64, 1024, 64), "classes": _size(rng, 2, 16, 2)}
    if kind == "block":
        return {"kind": kind, "batch": _size(rng, 1, 8, 2), "seq": _size(rng, 32, 1024, 64),
                "width": 64 * _size(rng, 4, 16, 4)}
    if kind == "dense":
        dtype = rng.choice(["f32", "f32", "f64"])
        return {"kind": kind, "m": _size(rng, 200, 8192, 64), "k": _size(rng, 100, 4096, 64),
                "n": _size(rng, 48, 4096, 64), "dtype": dtype}
    if kind == "heads":
        return {"kind": kind, "batch": _size(rng, 1, 8, 2), "heads": _size(rng, 4, 16, 4),
                "seq": _size(rng, 64, 1024, 64), "dh": rng.choice([64, 64, 96, 128]),
                "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "softmax":
        n = _size(rng, 32, 50000, 64)
        return {"kind": kind, "rows": _size(rng, max(8, 400000 // n), 20000000 // n), "n": n,
                "dtype": rng.choice(["f32", "f32", "f64"])}
    if kind == "layernorm":
        n = _size(rng, 128, 8192, 64)
        return {"kind": kind, "rows": _size(rng, 200, 20000000 // n), "n": n, "dtype": rng.choice(["f32", "f32", "f64"])}
    if kind == "embed":
        return {"kind": kind, "tokens": _size(rng, 500, 32768, 64), "vocab": _size(rng, 1000, 64000, 64),
                "width": _size(rng, 32, 1024, 32)}
    return {"kind": kind, "n": _size(rng, 1000, 50000, 64), "d": _size(rng, 8, 4096, 8),
            "dtype": rng.choice(["f32", "f32", "f64"])}


def _cost(case):
    w = work(case)
    rate = {"f64": 5e13, "bf16": 1e15, "f16": 1e15}.get(case.get("dtype"), 1e14)
    return w["bytes"] / 4e12 + w["flops"] / rate


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _drawn(rng)
        if _cost(case) <= most:
            return case


# ---------------------------------------------------------------- inputs
def _tensors(case, seed):
    """The case's inputs on the GPU, by name, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + 17)
    kind, dt = case["kind"], TORCH[case.get("dtype", "f32")]

    def normal(*shape, scale=1.0, dtype=dt):
        draws = torch.float64 if dtype == torch.float64 else torch.float32
        return (torch.randn(*shape, generator=g, device="cuda", dtype=draws) * scale).to(dtype)

    if kind == "linreg":
        X, w = normal(case["n"], case["d"]), normal(case["d"])
        return {"X": X, "w": normal(case["d"]), "y": X @ w + normal(case["n"], scale=0.01)}
    if kind == "mlp":
        b, i, h, o = case["batch"], case["d_in"], case["hidden"], case["classes"]
        labels = torch.randint(0, o, (b,), generator=g, device="cuda")
        return {"x": torch.rand(b, i, generator=g, device="cuda"),
                "onehot": torch.nn.functional.one_hot(labels, o).float(), "w1": normal(i, h, scale=math.sqrt(2 / i)),
                "b1": normal(h, scale=0.01), "w2": normal(h, o, scale=math.sqrt(2 / h)), "b2": normal(o, scale=0.01)}
    if kind == "block":
        b, s, d = case["batch"], case["seq"], case["width"]
        t = {"x": normal(b, s, d), "g1": 1 + normal(d, scale=0.1), "c1": normal(d, scale=0.1)}
        for name in ("q", "k", "v", "o"):
            t["w" + name], t["b" + name] = normal(d, d, scale=0.02), normal(d, scale=0.02)
        t.update(g2=1 + normal(d, scale=0.1), c2=normal(d, scale=0.1), wf=normal(d, 4 * d, scale=0.02),
                 bf=normal(4 * d, scale=0.02), wp=normal(4 * d, d, scale=0.02), bp=normal(d, scale=0.02))
        return t
    if kind == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        return {"x": normal(m, k), "w": normal(k, n, scale=1 / math.sqrt(k)), "b": normal(n, scale=0.1),
                "g": normal(m, n, scale=0.01)}
    if kind == "heads":
        b, h, s, e = case["batch"], case["heads"], case["seq"], case["dh"]
        scores = torch.randn(b, h, s, s, generator=g, device="cuda")
        return {"q": normal(b, s, h, e), "k": normal(b, s, h, e), "v": normal(b, s, h, e),
                "p": torch.softmax(scores, -1).to(dt)}
    if kind == "softmax":
        return {"x": normal(case["rows"], case["n"], scale=2.0), "g": normal(case["rows"], case["n"])}
    if kind == "layernorm":
        n = case["n"]
        return {"x": normal(case["rows"], n) * 1.5 + 0.25, "gamma": 1 + normal(n, scale=0.1), "beta": normal(n, scale=0.1)}
    if kind == "embed":
        # log-uniform ids: the frequencies of a vocabulary sorted by rank
        u = torch.rand(case["tokens"], generator=g, device="cuda", dtype=torch.float64)
        ids = (torch.exp(u * math.log(case["vocab"] + 1)) - 1).long().clamp_(0, case["vocab"] - 1)
        return {"table": normal(case["vocab"], case["width"], scale=0.02), "ids": ids,
                "g": normal(case["tokens"], case["width"], scale=0.01)}
    return {"x": normal(case["n"], case["d"]) * 3.0 + 1.0}


def _results(case):
    """name -> (shape, dtype) of the case's results."""
    kind, dt = case["kind"], case.get("dtype", "f32")
    if kind == "linreg":
        return {"grad": ((case["d"],), dt), "loss": ((), dt)}
    if kind == "mlp":
        i, h, o = case["d_in"], case["hidden"], case["classes"]
        return {"loss": ((), dt), "w1": ((i, h), dt), "b1": ((h,), dt), "w2": ((h, o), dt), "b2": ((o,), dt)}
    if kind == "block":
        return {"y": ((case["batch"], case["seq"], case["width"]), dt)}
    if kind == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        return {"y": ((m, n), dt), "dx": ((m, k), dt), "dw": ((k, n), dt), "db": ((n,), dt)}
    if kind == "heads":
        b, h, s, e = case["batch"], case["heads"], case["seq"], case["dh"]
        return {"scores": ((b, h, s, s), dt), "o": ((b, h, s, e), dt)}
    if kind == "softmax":
        return {"y": ((case["rows"], case["n"]), dt), "dx": ((case["rows"], case["n"]), dt)}
    if kind == "layernorm":
        return {"y": ((case["rows"], case["n"]), dt)}
    if kind == "embed":
        return {"rows": ((case["tokens"], case["width"]), dt), "table": ((case["vocab"], case["width"]), dt)}
    n, d = case["n"], case["d"]
    return {"mean": ((d,), dt), "var": ((d,), dt), "y": ((n, d), dt)}


def _wrap(t):
    """A torch tensor's storage as a borrowed device tensor of the library."""
    name = {torch.float32: "f32", torch.float64: "f64", torch.bfloat16: "bf16", torch.float16: "f16",
            torch.int64: "i64"}[t.dtype]
    return C.borrow(tuple(t.shape), NP[name], t.data_ptr(), t.numel() * t.element_size())


def prepare(case, seed):
    held = {k: v.contiguous() for k, v in _tensors(case, seed).items()}
    out = {k: torch.zeros(shape, dtype=TORCH[dt], device="cuda") for k, (shape, dt) in _results(case).items()}
    s = {"kind": case["kind"], "held": held, "out": out}
    i = s["in"] = {k: _wrap(v) for k, v in held.items()}
    o = s["to"] = {k: _wrap(v) for k, v in out.items()}
    if case["kind"] == "mlp":
        s["key"] = C.key_tensor(KEY + seed)
    elif case["kind"] == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        s["xt"], s["wt"] = i["x"].view((k, m), (1, k)), i["w"].view((n, k), (1, n))
    elif case["kind"] == "heads":
        b, h, q, e = case["batch"], case["heads"], case["seq"], case["dh"]
        st = (q * h * e, e, h * e, 1)
        s["q"], s["v"] = i["q"].view((b, h, q, e), st), i["v"].view((b, h, q, e), st)
        s["kt"] = i["k"].view((b, h, e, q), (st[0], st[1], 1, st[2]))
    elif case["kind"] == "standardise":
        n, d = case["n"], case["d"]
        s["mean"], s["var"] = o["mean"].view((n, d), (0, 1)), o["var"].view((n, d), (0, 1))
        s["by_n"] = C.fused_chain([("const", 0, 0, float(n)), ("div", 0, ("s", 0))])
        s["square"] = C.fused_chain([("sub", 0, 1), ("mul", ("s", 0), ("s", 0))])
        s["scale"] = C.fused_chain([("sub", 0, 1), ("const", 0, 0, EPS), ("add", 2, ("s", 1)), ("sqrt", ("s", 2)),
                                    ("div", ("s", 0), ("s", 3))])
    # the library works on its own stream: what torch has in flight is finished first
    torch.cuda.synchronize()
    return s


def run(s):
    kind, i, o = s["kind"], s["in"], s["to"]
    if kind == "linreg":
        C.program("linreg_step", [i["X"], i["w"], i["y"]], [o["grad"], o["loss"]])
    elif kind == "mlp":
        C.program("mlp_train_step", [i["x"], i["onehot"], i["w1"], i["b1"], i["w2"], i["b2"], s["key"]],
                  [o["loss"], o["w1"], o["b1"], o["w2"], o["b2"]])
    elif kind == "block":
        C.program("transformer_block", [i[k] for k in ("x", "g1", "c1", "wq", "bq", "wk", "bk", "wv", "bv", "wo", "bo",
                                                       "g2", "c2", "wf", "bf", "wp", "bp")], [o["y"]])
    elif kind == "dense":
        C.linear(i["x"], i["w"], bias=i["b"], act="relu", c=o["y"])
        C.matmul(i["g"], s["wt"], c=o["dx"])
        C.matmul(s["xt"], i["g"], c=o["dw"])
        C.reduce("sum", i["g"], 0, out=o["db"])
    elif kind == "heads":
        C.matmul(s["q"], s["kt"], c=o["scores"])
        C.matmul(i["p"], s["v"], c=o["o"])
    elif kind == "softmax":
        C.softmax(i["x"], o["y"])
        C.softmax_adjoint(o["y"], i["g"], o["dx"])
    elif kind == "layernorm":
        C.layer_norm(i["x"], i["gamma"], i["beta"], EPS, o["y"])
    elif kind == "embed":
        C.gather(i["table"], i["ids"], 0, out=o["rows"], deferred=True)
        C.scatter(i["table"], i["ids"], i["g"], 0, add=True, out=o["table"], deferred=True)
    else:
        C.reduce("sum", i["x"], 0, out=o["mean"])
        C.fused_elementwise(s["by_n"], [o["mean"]], o["mean"])
        C.reduce("sum", [i["x"], s["mean"]], 0, out=o["var"], chain=s["square"])
        C.fused_elementwise(s["by_n"], [o["var"]], o["var"])
        C.fused_elementwise(s["scale"], [i["x"], s["mean"], s["var"]], o["y"])
    return s["out"]


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind, w = case["kind"], WIDTH[case.get("dtype", "f32")]
    if kind == "linreg":
        n, d = case["n"], case["d"]
        return {"bytes": w * (n * d + n + 2 * d + 1), "flops": 4 * n * d + 3 * n}
    if kind == "mlp":
        b, i, h, o = case["batch"], case["d_in"], case["hidden"], case["classes"]
        return {"bytes": w * (b * i + b * o + 2 * (i * h + h + h * o + o)),
                "flops": 4 * b * i * h + 6 * b * h * o + 2 * i * h}
    if kind == "block":
        b, s, d = case["batch"], case["seq"], case["width"]
        return {"bytes": w * (2 * b * s * d + 12 * d * d + 13 * d),
                "flops": 24 * b * s * d * d + 2 * b * s * (s + 1) * d}
    if kind == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": w * (2 * m * k + 2 * k * n + 2 * m * n + 2 * n), "flops": 6 * m * k * n + 3 * m * n}
    if kind == "heads":
        b, h, s, e = case["batch"], case["heads"], case["seq"], case["dh"]
        return {"bytes": w * b * h * (4 * s * e + 2 * s * s), "flops": 4 * b * h * s * s * e}
    if kind == "softmax":
        return {"bytes": 4 * w * case["rows"] * case["n"], "flops": 9 * case["rows"] * case["n"]}
    if kind == "layernorm":
        return {"bytes": w * (2 * case["rows"] * case["n"] + 2 * case["n"]), "flops": 8 * case["rows"] * case["n"]}
    if kind == "embed":
        t, v, d = case["tokens"], case["vocab"], case["width"]
        return {"bytes": w * (3 * t * d + 2 * v * d) + 8 * t, "flops": t * d}
    n, d = case["n"], case["d"]
    return {"bytes": w * (2 * n * d + 2 * d), "flops": 6 * n * d}


def tolerance(case):
    kind, dt = case["kind"], case.get("dtype", "f32")
    if kind == "heads":
        # binary32 sums stored once at 16 bits: one rounding unit, more where two sums straddle a rounding line
        return {"rel": 2e-3 if dt == "bf16" else 3e-4}
    if kind == "block":
        return {"rel": 4e-6}
    if dt == "f64":
        return {"rel": 1e-13}
    return {"rel": 4e-6 if kind == "dense" else 2e-6}


# ---------------------------------------------------------------- the same in 64 bits
def _keep(key, count):
    """The dropout mask of `count` elements: unit(word(key, i)) >= rate at
    binary32, word = splitmix64(key ^ rotl(splitmix64(i), 41))."""
    def mix(x):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))

    with np.errstate(over="ignore"):
        j = mix(np.arange(count, dtype=np.uint64))
        word = mix(np.uint64(key) ^ ((j << np.uint64(41)) | (j >> np.uint64(23))))
    unit = ((word >> np.uint64(11)).astype(np.float64) * 2.0 ** -53).astype(np.float32)
    return torch.from_numpy(unit >= np.float32(RATE))


def _norm(x, gamma, beta):
    c = x - x.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + EPS) * gamma + beta


def exact(case, seed):
    kind = case["kind"]
    raw = _tensors(case, seed)
    t = {k: v if v.dtype == torch.int64 else v.double() for k, v in raw.items()}
    if kind == "linreg":
        r = t["X"] @ t["w"] - t["y"]
        return {"grad": t["X"].T @ r / case["n"], "loss": (r * r).mean()}
    if kind == "mlp":
        b, h = case["batch"], case["hidden"]
        rate, lr = float(np.float32(RATE)), float(np.float32(LEARN))
        keep = _keep(KEY + seed, b * h).reshape(b, h).cuda().double() / float(np.float32(1) - np.float32(rate))
        z1 = t["x"] @ t["w1"] + t["b1"]
        d = z1.clamp_min(0) * keep
        z2 = d @ t["w2"] + t["b2"]
        logp = torch.log_softmax(z2, 1)
        gz2 = (logp.exp() - t["onehot"]) / b
        gz1 = (gz2 @ t["w2"].T) * keep * (z1 > 0)
        return {"loss": -(logp * t["onehot"]).sum(1).mean(), "w1": t["w1"] - lr * (t["x"].T @ gz1),
                "b1": t["b1"] - lr * gz1.sum(0), "w2": t["w2"] - lr * (d.T @ gz2), "b2": t["b2"] - lr * gz2.sum(0)}
    if kind == "block":
        b, s, d = case["batch"], case["seq"], case["width"]
        x = t["x"]
        h = _norm(x, t["g1"], t["c1"])
        q, k, v = ((h @ t["w" + n] + t["b" + n]).reshape(b, s, d // HEAD, HEAD).transpose(1, 2).contiguous()
                   for n in "qkv")
        a = (q @ k.transpose(2, 3).contiguous()) * HEAD ** -0.5
        a = a.masked_fill(torch.ones(s, s, dtype=torch.bool, device="cuda").triu(1), -math.inf)
        x = x + (torch.softmax(a, -1) @ v).transpose(1, 2).reshape(b, s, d) @ t["wo"] + t["bo"]
        f = _norm(x, t["g2"], t["c2"]) @ t["wf"] + t["bf"]
        return {"y": x + (f * 0.5 * torch.special.erfc(-f * math.sqrt(0.5))) @ t["wp"] + t["bp"]}
    if kind == "dense":
        return {"y": (t["x"] @ t["w"] + t["b"]).clamp_min(0), "dx": t["g"] @ t["w"].T, "dw": t["x"].T @ t["g"],
                "db": t["g"].sum(0)}
    if kind == "heads":
        q, k, v = (t[n].transpose(1, 2).contiguous() for n in "qkv")
        return {"scores": q @ k.transpose(2, 3).contiguous(), "o": t["p"] @ v}
    if kind == "softmax":
        y = torch.softmax(t["x"], -1)
        return {"y": y, "dx": y * (t["g"] - (t["g"] * y).sum(-1, keepdim=True))}
    if kind == "layernorm":
        return {"y": _norm(t["x"], t["gamma"], t["beta"])}
    if kind == "embed":
        return {"rows": t["table"][t["ids"]], "table": t["table"].index_add(0, t["ids"], t["g"])}
    mean, var = t["x"].mean(0), t["x"].var(0, unbiased=False)
    return {"mean": mean, "var": var, "y": (t["x"] - mean) / torch.sqrt(var + EPS)}
