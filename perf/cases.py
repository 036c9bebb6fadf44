"""The work that a program using this framework has it do, as cases that can be timed and checked.

A case is a dict of plain values: a "kind" (which of the op sequences below it runs), its sizes and its options. Every
kind runs forward and, unless it says otherwise, backward, through the package's public calls, with the gradients in
buffers that an optimizer would keep. Sizes are those of this repository's benchmark and tests, or generic ones
between them.

  matmul      C = A B, with train also dA = G B^T and dB = A^T G
  mlp         three linear layers with ReLU between, and their backward
  conv        conv2d_relu, with pool followed by a 2 x 2 max pool, and the backward of both
  attention   softmax(Q K^T / sqrt(Dh)) V over heads with the probabilities kept, and its backward
  layernorm   over the last axis, and its backward
  batchnorm   training-mode statistics with the folded ReLU, and its backward
  block       a pre-norm transformer block (attention and a GELU MLP, both with residuals), and its backward
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "nn-cpp_amd"))

import nnh  # noqa: E402

EPS = 1e-5


def listed():
    return [
        # A small square layer product, trained: three products (NN, NT, TN) too small to fill the chip for long, where
        # latency and launches count.
        {"name": "matmul_512_train", "kind": "matmul", "m": 512, "n": 512, "k": 512, "train": True},
        # Sizes that no tile divides, rows that are not 16-byte aligned: a product of a program that pads nothing.
        {"name": "matmul_ragged_train", "kind": "matmul", "m": 1021, "n": 771, "k": 1533, "train": True},
        # A few rows against a large weight, as inference over a small batch has them.
        {"name": "matmul_64x4096x4096", "kind": "matmul", "m": 64, "n": 4096, "k": 4096, "train": False},
        # The large product that the benchmark's headline is quoted on.
        {"name": "matmul_4096", "kind": "matmul", "m": 4096, "n": 4096, "k": 4096, "train": False},
        # The image classifier's MLP, one training step's layers at its usual batch.
        {"name": "mlp_256", "kind": "mlp", "batch": 256, "d0": 784, "d1": 512, "d2": 256, "d3": 10},
        # A CNN's first layer: one input channel, all memory traffic.
        {"name": "conv_first", "kind": "conv", "n": 128, "cin": 1, "h": 28, "w": 28, "cout": 32, "kernel": 3, "stride": 1,
         "pad": 1, "pool": True},
        # Its second layer: the contraction that dominates such a network.
        {"name": "conv_second", "kind": "conv", "n": 128, "cin": 32, "h": 14, "w": 14, "cout": 64, "kernel": 3,
         "stride": 1, "pad": 1, "pool": True},
        # Self-attention at a training batch.
        {"name": "attention_256", "kind": "attention", "n": 32, "tq": 256, "tk": 256, "heads": 8, "dh": 64,
         "causal": False, "mask": False},
        # The same model's normalisation over every token of the batch.
        {"name": "layernorm_8192x512", "kind": "layernorm", "rows": 8192, "d": 512},
        # A CNN's batch norm after its first convolution.
        {"name": "batchnorm_48", "kind": "batchnorm", "n": 64, "c": 16, "h": 48, "w": 48},
        # A small causal language model's block: about thirty short calls, the least work of the list.
        {"name": "block_64", "kind": "block", "n": 16, "t": 64, "heads": 4, "dh": 16, "causal": True},
        # A block of ordinary width at a training batch, where everything above meets.
        {"name": "block_512", "kind": "block", "n": 32, "t": 256, "heads": 8, "dh": 64, "causal": True},
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _some(rng, lo, hi):
    """A size between lo and hi over the logarithm: half of them as they come, half multiples of 16."""
    v = _logint(rng, lo, hi)
    return v if rng.random() < 0.5 or v < 32 else v // 16 * 16


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "mlp", "conv", "conv", "attention", "layernorm", "batchnorm", "block"])
    if kind == "matmul":
        c = {"kind": kind, "m": _some(rng, 48, 4096), "n": _some(rng, 48, 4096), "k": _some(rng, 48, 4096),
             "train": rng.random() < 0.6}
        c["train"] = c["train"] and c["m"] * c["n"] * c["k"] < 2e10  # three products cost no more than the largest one
    elif kind == "mlp":
        c = {"kind": kind, "batch": _some(rng, 24, 4096), "d0": _some(rng, 64, 1024), "d1": _some(rng, 48, 1024),
             "d2": _some(rng, 48, 1024), "d3": rng.randint(2, 64)}
    elif kind == "conv":
        kernel = rng.choice([3, 3, 3, 5])
        side = rng.choice([14, 16, 28, 32, 48, rng.randint(9, 48)])
        cin, cout = rng.choice([(1, 8), (1, 16), (1, 32), (3, 16), (3, 32), (8, 16), (16, 32), (32, 64), (24, 40), (64, 64)])
        n = _logint(rng, 8, min(256, max(16, int(6e9 / (2.0 * cin * cout * kernel * kernel * side * side)))))
        c = {"kind": kind, "n": n, "cin": cin, "h": side, "w": rng.choice([side, side, rng.randint(9, 48)]),
             "cout": cout, "kernel": kernel, "stride": rng.choice([1, 1, 1, 2]),
             "pad": rng.choice([kernel // 2, kernel // 2, 0]), "pool": rng.random() < 0.6}
    elif kind == "attention":
        tq = _some(rng, 16, 512)
        tk = tq if rng.random() < 0.8 else _some(rng, 16, 512)
        heads = rng.choice([2, 4, 8])
        c = {"kind": kind, "n": _logint(rng, 1, max(1, min(64, int(32 * 8 * 256 * 256 / (heads * tq * tk))))), "tq": tq,
             "tk": tk, "heads": heads, "dh": rng.choice([16, 32, 64, 64, 80]), "causal": tq == tk and rng.random() < 0.6,
             "mask": rng.random() < 0.3}
    elif kind == "layernorm":
        d = _some(rng, 32, 1024)
        c = {"kind": kind, "rows": _some(rng, 64, min(32768, 8192 * 1024 // d)), "d": d}
    elif kind == "batchnorm":
        side = rng.randint(5, 48)
        ch = rng.choice([8, 16, 24, 32, 64])
        c = {"kind": kind, "n": _logint(rng, 8, max(8, min(128, int(4e6 / (ch * side * side))))), "c": ch, "h": side,
             "w": side}
    else:
        t = _some(rng, 32, 256)
        heads, dh = rng.choice([(2, 32), (4, 16), (4, 32), (4, 64), (8, 32), (8, 64)])
        c = {"kind": kind, "n": _logint(rng, 4, max(4, min(64, 8192 // t))), "t": t, "heads": heads, "dh": dh,
             "causal": rng.random() < 0.7}
    return c


# ---- inputs ----

class _Inputs:
    """Seeded draws on the GPU, the same for prepare and exact."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def uniform(self, *shape, lo=-1.0, hi=1.0):
        return torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda")

    def weight(self, *shape):
        """U(+-1/sqrt(fan_in)), as the modules initialise their weights."""
        bound = 1.0 / math.sqrt(math.prod(shape[1:]))
        return self.uniform(*shape, lo=-bound, hi=bound)


def _conv_out(c):
    return tuple((s + 2 * c["pad"] - c["kernel"]) // c["stride"] + 1 for s in (c["h"], c["w"]))


_BLOCK_WEIGHTS = ("wq", "wk", "wv", "wo", "w1", "w2")


def _tensors(c, seed):
    """The case's inputs by name."""
    i, kind = _Inputs(seed), c["kind"]
    if kind == "matmul":
        t = {"a": i.uniform(c["m"], c["k"]), "b": i.uniform(c["k"], c["n"])}
        if c["train"]:
            t["g"] = i.normal(c["m"], c["n"])
    elif kind == "mlp":
        d = [c["d0"], c["d1"], c["d2"], c["d3"]]
        t = {"x": i.uniform(c["batch"], d[0], lo=0.0), "g": i.normal(c["batch"], d[3])}
        for k in range(3):
            t["w%d" % k], t["b%d" % k] = i.weight(d[k + 1], d[k]), 0.1 * i.normal(d[k + 1])
    elif kind == "conv":
        ho, wo = _conv_out(c)
        if c["pool"]:
            ho, wo = ho // 2, wo // 2
        t = {"x": i.uniform(c["n"], c["cin"], c["h"], c["w"], lo=0.0),
             "w": i.weight(c["cout"], c["cin"], c["kernel"], c["kernel"]), "b": 0.1 * i.normal(c["cout"]),
             "g": i.normal(c["n"], c["cout"], ho, wo)}
    elif kind == "attention":
        d = c["heads"] * c["dh"]
        t = {"q": i.normal(c["n"], c["tq"], d), "k": i.normal(c["n"], c["tk"], d), "v": i.normal(c["n"], c["tk"], d),
             "g": i.normal(c["n"], c["tq"], d)}
        if c["mask"]:  # sequences of different lengths, none empty
            live = torch.randint(1, c["tk"] + 1, (c["n"], 1), generator=i.gen, device="cuda")
            t["mask"] = (torch.arange(c["tk"], device="cuda")[None, :] < live).float()
    elif kind == "layernorm":
        t = {"x": i.normal(c["rows"], c["d"]), "gamma": 1.0 + 0.1 * i.normal(c["d"]), "beta": 0.1 * i.normal(c["d"]),
             "g": i.normal(c["rows"], c["d"])}
    elif kind == "batchnorm":
        shape = (c["n"], c["c"], c["h"], c["w"])
        t = {"x": i.normal(*shape) + 0.5, "w": 1.0 + 0.1 * i.normal(c["c"]), "b": 0.1 * i.normal(c["c"]),
             "g": i.normal(*shape)}
    else:
        d = c["heads"] * c["dh"]
        t = {"x": i.normal(c["n"], c["t"], d), "g": i.normal(c["n"], c["t"], d)}
        for k in ("1", "2"):
            t["gamma" + k], t["beta" + k] = 1.0 + 0.1 * i.normal(d), 0.1 * i.normal(d)
        for name, rows, cols in (("q", d, d), ("k", d, d), ("v", d, d), ("o", d, d), ("1", 4 * d, d), ("2", d, 4 * d)):
            t["w" + name], t["b" + name] = i.weight(rows, cols), 0.1 * i.normal(rows)
    return t


_GRADIENTS = {"matmul": ("a", "b"), "mlp": ("x", "w0", "b0", "w1", "b1", "w2", "b2"), "conv": ("x", "w", "b"),
              "attention": ("q", "k", "v"), "layernorm": ("x", "gamma", "beta"), "batchnorm": ("x", "w", "b"),
              "block": ("x", "gamma1", "beta1", "gamma2", "beta2") + _BLOCK_WEIGHTS +
                       tuple("b" + w[1:] for w in _BLOCK_WEIGHTS)}


def prepare(case, seed):
    s = _tensors(case, seed)
    s["case"] = case
    if case.get("train", True):
        s["d"] = {k: torch.empty_like(s[k]) for k in _GRADIENTS[case["kind"]]}
    if case["kind"] == "mlp":  # the hidden layers' gradients
        s["dh"] = [torch.empty(case["batch"], case["d%d" % k], device="cuda") for k in (1, 2)]
    if case["kind"] == "conv":
        s["dy"] = torch.empty((case["n"], case["cout"]) + _conv_out(case), device="cuda") if case["pool"] else None
    if case["kind"] == "block":  # the activations' gradients
        x = s["x"]
        s["da"] = {k: torch.empty_like(x) for k in ("n1", "q", "k", "v", "att", "h", "n2")}
        s["da"]["f"] = torch.empty(*x.shape[:2], 4 * x.shape[2], device="cuda")
        s["da"]["m"] = torch.empty_like(s["da"]["f"])
    return s


# ---- one pass ----

def _ptr(t):
    return t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _run_matmul(s):
    y = nnh.matmul(s["a"], s["b"])
    if "g" not in s:
        return {"y": y}
    nnh.matmul_backward(s["g"], s["a"], s["b"], da=s["d"]["a"], db=s["d"]["b"])
    return {"y": y, "d": s["d"]}


def _run_mlp(s):
    d = s["d"]
    h0 = nnh.linear_forward(s["x"], s["w0"], s["b0"], relu=True)
    h1 = nnh.linear_forward(h0, s["w1"], s["b1"], relu=True)
    y = nnh.linear_forward(h1, s["w2"], s["b2"])
    dh0, dh1 = s["dh"]
    nnh.linear_backward(s["g"], h1, s["w2"], dx=dh1, dw=d["w2"], db=d["b2"])
    nnh.relu_backward(h1, dh1, dh1)
    nnh.linear_backward(dh1, h0, s["w1"], dx=dh0, dw=d["w1"], db=d["b1"])
    nnh.relu_backward(h0, dh0, dh0)
    nnh.linear_backward(dh0, s["x"], s["w0"], dx=d["x"], dw=d["w0"], db=d["b0"])
    return {"y": y, "d": d}


def _run_conv(s):
    c, d, g = s["case"], s["d"], s["g"]
    if c["pool"]:
        y, alive, pooled, argmax = nnh.conv2d_relu_maxpool2d_forward(s["x"], s["w"], s["b"], c["stride"], c["pad"], 2, 2)
        nnh.check(nnh.lib().nnh_maxpool2d_backward(_ptr(g), _ptr(argmax), *y.shape, 2, 2, _ptr(s["dy"]), 1, _stream()))
        g = s["dy"]
        out = {"y": y, "alive": alive, "pooled": pooled, "argmax": argmax}
    else:
        y, alive = nnh.conv2d_forward(s["x"], s["w"], s["b"], c["stride"], c["pad"], True)
        out = {"y": y, "alive": alive}
    nnh.conv2d_backward(g, s["x"], s["w"], alive, c["stride"], c["pad"], dx=d["x"], dw=d["w"], db=d["b"])
    out["d"] = d
    return out


def _run_attention(s):
    c, d = s["case"], s["d"]
    out, probs = nnh.attention_forward(s["q"], s["k"], s["v"], c["heads"], mask=s.get("mask"), causal=c["causal"])
    nnh.attention_backward(s["g"], s["q"], s["k"], s["v"], probs, c["heads"], mask=s.get("mask"), causal=c["causal"],
                           dq=d["q"], dk=d["k"], dv=d["v"])
    return {"out": out, "probs": probs, "d": d}


def _run_layernorm(s):
    d = s["d"]
    y, mean, inv = nnh.layernorm_forward(s["x"], s["gamma"], s["beta"], EPS)
    nnh.layernorm_backward(s["g"], s["x"], s["gamma"], mean, inv, dx=d["x"], dgamma=d["gamma"], dbeta=d["beta"])
    return {"y": y, "mean": mean, "inv": inv, "d": d}


def _run_batchnorm(s):
    d = s["d"]
    y, alive, mean, var, inv = nnh.batchnorm_forward(s["x"], s["w"], s["b"], EPS, fuse_relu=True)
    nnh.batchnorm_backward(s["g"], s["x"], alive, s["w"], mean, inv, dx=d["x"], dw=d["w"], db=d["b"])
    return {"y": y, "alive": alive, "mean": mean, "var": var, "inv": inv, "d": d}


def _run_block(s):
    c, d, da, L, st = s["case"], s["d"], s["da"], nnh.lib(), _stream()
    x, g, heads, causal = s["x"], s["g"], c["heads"], c["causal"]
    n1, mean1, inv1 = nnh.layernorm_forward(x, s["gamma1"], s["beta1"], EPS)
    q, k, v = nnh.linear_forward_multi(n1, [(s["wq"], s["bq"]), (s["wk"], s["bk"]), (s["wv"], s["bv"])])
    att, probs = nnh.attention_forward(q, k, v, heads, causal=causal)
    h = nnh.linear_forward_add(att, s["wo"], s["bo"], x)
    n2, mean2, inv2 = nnh.layernorm_forward(h, s["gamma2"], s["beta2"], EPS)
    tokens, D = x.shape[0] * x.shape[1], x.shape[2]
    f, m, tanh = (torch.empty(*x.shape[:2], 4 * D, device=x.device) for _ in range(3))
    nnh.check(L.nnh_linear_gelu_forward(_ptr(n2), tokens, D, _ptr(s["w1"]), 4 * D, _ptr(s["b1"]), _ptr(f), _ptr(m),
                                        _ptr(tanh), st))
    y = nnh.linear_forward_add(m, s["w2"], s["b2"], h)
    # backward, last op first; a gradient that two ops write is stored by the first and added to by the second
    nnh.linear_backward(g, m, s["w2"], dx=da["m"], dw=d["w2"], db=d["b2"])
    nnh.check(L.nnh_gelu_backward(_ptr(f), _ptr(tanh), _ptr(da["m"]), f.numel(), _ptr(da["f"]), 1, st))
    nnh.linear_backward(da["f"], n2, s["w1"], dx=da["n2"], dw=d["w1"], db=d["b1"])
    nnh.check(L.nnh_add_to_grad(_ptr(da["h"]), _ptr(g), g.numel(), 1, st))
    nnh.layernorm_backward(da["n2"], h, s["gamma2"], mean2, inv2, dx=da["h"], dx_first=False, dgamma=d["gamma2"],
                           dbeta=d["beta2"])
    nnh.linear_backward(da["h"], att, s["wo"], dx=da["att"], dw=d["wo"], db=d["bo"])
    nnh.attention_backward(da["att"], q, k, v, probs, heads, causal=causal, dq=da["q"], dk=da["k"], dv=da["v"])
    nnh.linear_backward(da["q"], n1, s["wq"], dx=da["n1"], dw=d["wq"], db=d["bq"])
    nnh.linear_backward(da["k"], n1, s["wk"], dx=da["n1"], dx_first=False, dw=d["wk"], db=d["bk"])
    nnh.linear_backward(da["v"], n1, s["wv"], dx=da["n1"], dx_first=False, dw=d["wv"], db=d["bv"])
    nnh.check(L.nnh_add_to_grad(_ptr(d["x"]), _ptr(da["h"]), x.numel(), 1, st))
    nnh.layernorm_backward(da["n1"], x, s["gamma1"], mean1, inv1, dx=d["x"], dx_first=False, dgamma=d["gamma1"],
                           dbeta=d["beta1"])
    # without the keys' bias: a constant added to a row's scores changes nothing, its gradient is zero but for rounding
    return {"y": y, "d": {k: z for k, z in d.items() if k != "bk"}}


_RUN = {"matmul": _run_matmul, "mlp": _run_mlp, "conv": _run_conv, "attention": _run_attention,
        "layernorm": _run_layernorm, "batchnorm": _run_batchnorm, "block": _run_block}


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ---- what a pass cannot do without ----

def work(case):
    c, kind = case, case["kind"]
    if kind == "matmul":
        m, n, k = c["m"], c["n"], c["k"]
        return {"flops": (6.0 if c["train"] else 2.0) * m * n * k,
                "bytes": 4.0 * ((2 * m * k + 2 * k * n + 2 * m * n) if c["train"] else (m * k + k * n + m * n))}
    if kind == "mlp":
        d = [c["d0"], c["d1"], c["d2"], c["d3"]]
        wt = sum(d[k] * d[k + 1] for k in range(3))
        return {"flops": 6.0 * c["batch"] * wt, "bytes": 4.0 * (2 * wt + c["batch"] * (2 * d[0] + 2 * d[3]))}
    if kind == "conv":
        ho, wo = _conv_out(c)
        out, kk = c["n"] * c["cout"] * ho * wo, c["cin"] * c["kernel"] ** 2
        pooled = c["n"] * c["cout"] * (ho // 2) * (wo // 2) if c["pool"] else 0
        return {"flops": 6.0 * out * kk,
                "bytes": 4.0 * (2 * c["n"] * c["cin"] * c["h"] * c["w"] + 2 * c["cout"] * kk + out) + out +
                         (12.0 * pooled if c["pool"] else 4.0 * out)}
    if kind == "attention":
        rows, keys, d = c["n"] * c["tq"], c["n"] * c["tk"], c["heads"] * c["dh"]
        live = 0.5 if c["causal"] else 1.0
        return {"flops": live * 12.0 * rows * c["tk"] * d,
                "bytes": 4.0 * (rows * d * 4 + keys * d * 4 + rows * c["tk"] * c["heads"])}
    if kind == "layernorm":
        return {"flops": 20.0 * c["rows"] * c["d"], "bytes": 4.0 * (4 * c["rows"] * c["d"] + 4 * c["d"] + 2 * c["rows"])}
    if kind == "batchnorm":
        e = c["n"] * c["c"] * c["h"] * c["w"]
        return {"flops": 20.0 * e, "bytes": 17.0 * e}
    d, tokens = c["heads"] * c["dh"], c["n"] * c["t"]
    return {"flops": 72.0 * tokens * d * d + (0.5 if c["causal"] else 1.0) * 12.0 * tokens * c["t"] * d,
            "bytes": 4.0 * (4 * tokens * d + 24 * d * d)}


def tolerance(case):
    # against 64 bits the outputs are off by 1e-7 (element-wise ops) to 2e-6 (sums over 8192 tokens or 4096 terms);
    # four times the most of that. Flags and window positions differ only where two values tie in 32 bits.
    return {"rel": 1e-5, "max": 1e-3, "differ": 1e-4}


# ---- the same outputs in 64 bits ----

def _exact_block(c, t):
    leaves = {k: t[k].requires_grad_() for k in _GRADIENTS["block"]}
    n, T, D, H = c["n"], c["t"], c["heads"] * c["dh"], c["heads"]
    x = leaves["x"]

    def norm(v, k):
        return F.layer_norm(v, (D,), leaves["gamma" + k], leaves["beta" + k], EPS)

    n1 = norm(x, "1")
    q, k, v = (F.linear(n1, leaves["w" + p], leaves["b" + p]) for p in "qkv")
    att, _ = _attention(q, k, v, H, c["causal"], None)
    h = x + F.linear(att, leaves["wo"], leaves["bo"])
    m = F.gelu(F.linear(norm(h, "2"), leaves["w1"], leaves["b1"]), approximate="tanh")
    y = h + F.linear(m, leaves["w2"], leaves["b2"])
    y.backward(t["g"])
    return {"y": y.detach(), "d": {k: p.grad for k, p in leaves.items() if k != "bk"}}


def _attention(q, k, v, heads, causal, mask):
    n, tq, d = q.shape
    tk = k.shape[1]
    q, k, v = (z.reshape(n, -1, heads, d // heads).transpose(1, 2).contiguous() for z in (q, k, v))
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(d // heads)
    if causal:
        s = s.masked_fill(torch.ones(tq, tk, dtype=torch.bool, device=s.device).triu(1), -math.inf)
    if mask is not None:
        s = s.masked_fill(mask[:, None, None, :] == 0, -math.inf)
    p = torch.softmax(s, -1)
    return torch.matmul(p, v).transpose(1, 2).reshape(n, tq, d), p


def exact(case, seed):
    c, kind = case, case["kind"]
    t = {k: v.double() for k, v in _tensors(c, seed).items()}
    if kind == "block":
        return _exact_block(c, t)
    if kind == "matmul":
        y = t["a"] @ t["b"]
        return {"y": y, "d": {"a": t["g"] @ t["b"].T, "b": t["a"].T @ t["g"]}} if c["train"] else {"y": y}
    leaves = {k: t[k].requires_grad_() for k in _GRADIENTS[kind]}
    if kind == "mlp":
        h = t["x"]
        for k in range(3):
            h = F.linear(h, t["w%d" % k], t["b%d" % k])
            h = torch.relu(h) if k < 2 else h
        out = {"y": h}
    elif kind == "conv":
        ho, wo = _conv_out(c)
        col = F.unfold(t["x"], c["kernel"], padding=c["pad"], stride=c["stride"])
        y = torch.relu(torch.matmul(t["w"].reshape(c["cout"], -1), col) + t["b"][:, None])
        y = y.reshape(c["n"], c["cout"], ho, wo)
        out = {"y": y, "alive": None}
        if c["pool"]:
            out = {"y": y, "alive": None, "pooled": F.max_pool2d(y, 2), "argmax": None}
    elif kind == "attention":
        o, p = _attention(t["q"], t["k"], t["v"], c["heads"], c["causal"], t.get("mask"))
        out = {"out": o, "probs": p}
    elif kind == "layernorm":
        mean = t["x"].mean(1)
        inv = torch.rsqrt(t["x"].var(1, unbiased=False) + EPS)
        y = (t["x"] - mean[:, None]) * inv[:, None] * t["gamma"] + t["beta"]
        out = {"y": y, "mean": mean, "inv": inv}
    else:
        mean, var = t["x"].mean((0, 2, 3)), t["x"].var((0, 2, 3), unbiased=False)
        inv = torch.rsqrt(var + EPS)
        y = torch.relu((t["x"] - mean[:, None, None]) * (t["w"] * inv)[:, None, None] + t["b"][:, None, None])
        out = {"y": y, "alive": None, "mean": mean, "var": var, "inv": inv}
    out[next(k for k in ("pooled", "out", "y") if k in out)].backward(t["g"])
    out = {k: None if v is None else v.detach() for k, v in out.items()}
    out["d"] = {k: v.grad for k, v in leaves.items()}
    return out
