"""The work that programs on this package give it, as timed cases.

A case is one call (or one forward and backward, or one optimizer step) through
the public entry points of ``novann_amd``: Linear products from one request to
a training batch, Conv2d blocks, pooling, quantization of whole tensors, the
optimizer step that re-quantizes a weight, and a small CNN from images to
logits.  ``listed()`` names twelve; ``draw(rng)`` gives others from the same
ranges.  ``exact`` restates each case in 64-bit torch arithmetic, with its own
quantizer, from the same seeded inputs.
"""
import numpy as np
import torch

from novann_amd import functional as F
from novann_amd import module as M
from novann_amd import optim, quant

LOGITS = 10          # classes of the small CNN
BN_EPS = 1e-5
ADAM = {"lr": 1e-3, "betas": (0.9, 0.999), "weight_decay": 1e-2}


# --------------------------------------------------------------------------
# the cases

def listed():
    return [
        # serving one request: a quantized 4096-wide layer applied to one row
        linear("linear 1 row", 1, 4096, 4096, "e4m3", "f32", True),
        # serving a small batch with FP4 weights on bf16 activations
        linear("linear 64 rows fp4", 64, 4096, 4096, "e2m1", "bf16", True),
        # an MLP's first layer over flattened 28 x 28 images, a ragged batch
        # and width
        linear("linear 1000x784x500", 1000, 784, 500, "e4m3", "f32", True),
        # the same layer in training: forward, then all three gradients
        linear("linear train 256x784x512", 256, 784, 512, "e4m3", "f32", True, train=True),
        # the headline Linear (4096 x 4096 E4M3, 2048 rows) in training
        linear("linear train 2048x4096x4096", 2048, 4096, 4096, "e4m3", "f32", True, train=True),
        # inference block of a strided stage: Conv2d + BatchNorm2d + ReLU on
        # bf16 activations, bf16 out
        conv("conv block 64-128 s2", 256, 64, 28, 28, 128, 3, 2, 1, "e4m3", "bf16", fused=True),
        # the second convolution of the MNIST pair in training (FP4 weights)
        conv("conv train 32-64 28x28", 256, 32, 28, 28, 64, 3, 1, 1, "e2m1", "f32", train=True),
        # a deeper stage in training: more channels than one LDS block holds
        conv("conv train 128-128 14x14", 64, 128, 14, 14, 128, 3, 1, 1, "e4m3", "f32",
             train=True),
        # quantizing and reading back a 256M-element tensor
        {"name": "quantize 256M e4m3", "op": "quantize", "n": 1 << 28, "src": "f32",
         "dtype": "e4m3"},
        # MaxPool2d 3 x 3 / 2 with padding in training: forward, then the input
        # gradient
        {"name": "maxpool train 3x3/2", "op": "maxpool", "n": 256, "c": 64, "h": 28, "w": 28,
         "k": 3, "s": 2, "p": 1, "x": "f32"},
        # one AdamW step on a 4096 x 4096 FP4 layer, codes and scale refreshed
        {"name": "adamw 4096x4096 fp4", "op": "adamw", "dout": 4096, "din": 4096,
         "dtype": "e2m1"},
        # classifying a batch of images: two fused Conv2d blocks, pools, Linear
        {"name": "cnn 64 images", "op": "cnn", "n": 64, "h": 28, "w": 28, "c1": 16, "c2": 32,
         "dtype": "e2m1"},
    ]


def linear(name, rows, din, dout, w, x, bias, train=False):
    return {"name": name, "op": "linear", "rows": rows, "din": din, "dout": dout, "wdtype": w,
            "xdtype": x, "bias": bias, "train": train}


def conv(name, n, c, h, w, co, k, s, p, wdtype, x, fused=False, train=False):
    return {"name": name, "op": "conv", "n": n, "c": c, "h": h, "w": w, "co": co, "k": k,
            "s": s, "p": p, "wdtype": wdtype, "xdtype": x, "fused": fused, "train": train}


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def _width(rng, lo, hi):
    """A layer width: mostly whole multiples of 16, 64 or 256, one in four odd
    or ragged."""
    v = _log(rng, lo, hi)
    step = rng.choice([1, 16, 64, 256])
    return v if v < 2 * step else v // step * step


def draw(rng):
    kind = rng.choice(["rows", "linear", "linear train", "conv", "conv train", "quantize",
                       "maxpool", "adamw", "cnn"])
    weight = rng.choice(["e4m3", "e5m2", "e2m1"])
    if kind == "rows":  # serving: few rows, wide layers
        c = linear("", _log(rng, 1, 64), _width(rng, 512, 4096), _width(rng, 512, 4096), weight,
                   rng.choice(["f32", "bf16"]), rng.random() < 0.5)
    elif kind in ("linear", "linear train"):
        train = kind == "linear train"
        c = linear("", _log(rng, 64, 2048), _width(rng, 64, 4096), _width(rng, 10, 4096), weight,
                   "f32" if train else rng.choice(["f32", "bf16"]), rng.random() < 0.75, train)
    elif kind in ("conv", "conv train"):
        train = kind == "conv train"
        fused = not train and rng.random() < 0.75
        k = rng.choice([1, 3, 3, 3, 5])
        side = _log(rng, 7, 56)
        # the channels of a stage grow as its maps shrink
        cmax = max(16, min(256, 64 * 28 // side))
        ch = rng.choice([1, 3, 16, 32, 64, 128, 256])
        ch = min(ch, cmax)
        co = min(rng.choice([16, 32, 48, 64, 128, 256]), cmax)
        n = _log(rng, 1, max(1, min(256, 2 * 256 * 64 * 784 // ((ch + co) * side * side))))
        c = conv("", n, ch, side, side + rng.choice([0, 0, 0, 1, 4]), co, k, rng.choice([1, 1, 2]),
                 k // 2, weight, "f32" if train else rng.choice(["f32", "bf16"]), fused, train)
    elif kind == "quantize":
        c = {"op": "quantize", "n": _log(rng, 1 << 16, 1 << 28) + rng.randrange(3),
             "src": rng.choice(["f32", "f32", "bf16"]), "dtype": weight}
    elif kind == "maxpool":
        k, s, p = rng.choice([(2, 2, 0), (3, 2, 1), (3, 1, 1), (3, 3, 0)])
        side = _log(rng, 7, 56)
        c = {"op": "maxpool", "n": _log(rng, 1, 256), "c": rng.choice([16, 32, 64]), "h": side,
             "w": side + rng.choice([0, 0, 1]), "k": k, "s": s, "p": p,
             "x": rng.choice(["f32", "bf16"])}
    elif kind == "adamw":
        c = {"op": "adamw", "dout": _width(rng, 10, 4096), "din": _width(rng, 64, 4096),
             "dtype": weight}
    else:
        side = rng.choice([28, 28, 32])
        c = {"op": "cnn", "n": _log(rng, 1, 256), "h": side, "w": side,
             "c1": rng.choice([16, 32]), "c2": rng.choice([32, 64]), "dtype": weight}
    c.pop("name", None)
    return c


# --------------------------------------------------------------------------
# inputs

class Inputs:
    """The tensors of a case, drawn on the GPU from its seed: the same for the
    package's calls and for ``exact``."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device=self.dev)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.gen, device=self.dev)

    def weight(self, *shape):
        """Kaiming-normal for ReLU."""
        return self.normal(*shape) * (2.0 / int(np.prod(shape[1:]))) ** 0.5

    def log_uniform(self, n):
        """Random signs, magnitudes log-uniform in [2^-20, 2^20]."""
        v = self.uniform(n).mul_(40.0).sub_(20.0).exp2_()
        return v.mul_(self.uniform(n).sub_(0.5).sign_())

    def bn(self, channels):
        """BatchNorm gamma, beta, running mean and variance after some training."""
        return (1.0 + 0.1 * self.normal(channels), 0.1 * self.normal(channels),
                0.1 * self.normal(channels), 0.5 + self.uniform(channels))


NARROW = {"f32": torch.float32, "bf16": torch.bfloat16}


def draws(case, seed):
    """The case's input tensors by name."""
    r, op = Inputs(seed), case["op"]
    t = {}
    if op == "linear":
        t["x"] = r.normal(case["rows"], case["din"]).to(NARROW[case["xdtype"]])
        t["w"] = r.weight(case["dout"], case["din"])
        if case["bias"]:
            t["b"] = 0.1 * r.normal(1, case["dout"])
        if case["train"]:
            t["g"] = r.normal(case["rows"], case["dout"])
    elif op == "conv":
        shape = (case["n"], case["c"], case["h"], case["w"])
        # images in [0, 1], or the activations of a ReLU
        x = r.uniform(*shape) if case["c"] <= 3 else r.normal(*shape).relu_()
        t["x"] = x.to(NARROW[case["xdtype"]])
        t["w"] = r.weight(case["co"], case["c"], case["k"], case["k"])
        t["b"] = 0.1 * r.normal(case["co"], 1)
        if case["fused"]:
            t["gamma"], t["beta"], t["mean"], t["var"] = r.bn(case["co"])
        if case["train"]:
            t["g"] = r.normal(case["n"], case["co"], *_out(case))
    elif op == "quantize":
        t["x"] = r.log_uniform(case["n"]).to(NARROW[case["src"]])
    elif op == "maxpool":
        t["x"] = r.normal(case["n"], case["c"], case["h"], case["w"]).relu_().to(
            NARROW[case["x"]])
        t["g"] = r.normal(case["n"], case["c"], *_out(case))
    elif op == "adamw":
        t["w"] = r.weight(case["dout"], case["din"])
        t["g"] = 0.01 * r.normal(case["dout"], case["din"])
    else:
        t["x"] = r.uniform(case["n"], 1, case["h"], case["w"])
        t["w1"], t["bn1"] = r.weight(case["c1"], 1, 3, 3), r.bn(case["c1"])
        t["w2"], t["bn2"] = r.weight(case["c2"], case["c1"], 3, 3), r.bn(case["c2"])
        t["w3"], t["b3"] = r.weight(LOGITS, case["c2"]), 0.1 * r.normal(1, LOGITS)
    return t


def _out(case):
    k, s, p = case["k"], case["s"], case["p"]
    return (case["h"] + 2 * p - k) // s + 1, (case["w"] + 2 * p - k) // s + 1


# --------------------------------------------------------------------------
# the package's side

def prepare(case, seed):
    t, op = draws(case, seed), case["op"]
    s = {"op": op, "case": case}
    if op in ("linear", "conv"):
        s["x"], s["g"] = t["x"], t.get("g")
        s["weight"] = M.QuantizedParameters.from_float(t["w"], case["wdtype"])
        s["bias"] = M.Parameters(t["b"]) if "b" in t else None
        if case.get("fused"):
            mul, add = _fold(t["gamma"], t["beta"], t["mean"], t["var"])
            s["epilogue"] = F.Epilogue(channel_mul=mul.float(), channel_add=add.float(),
                                       relu=True, out_dtype=case["xdtype"])
    elif op == "quantize":
        s["x"] = t["x"]
    elif op == "maxpool":
        s["x"], s["g"] = t["x"], t["g"]
        s["layer"] = M.MaxPool2d(case["k"], case["s"], case["p"])
    elif op == "adamw":
        s["weight"] = M.QuantizedParameters.from_float(t["w"], case["dtype"], keep_master=True)
        s["g"] = t["g"]
        s["opt"] = optim.AdamW([s["weight"]], **ADAM)
    else:
        s["x"] = t["x"]
        blocks = []
        for w, (gamma, beta, mean, var), stride in ((t["w1"], t["bn1"], 1),
                                                    (t["w2"], t["bn2"], 2)):
            layer = M.Conv2d(w.shape[1], w.shape[0], 3, stride=stride, padding=1, bias=False)
            layer.weight = M.QuantizedParameters.from_float(w, case["dtype"])
            bn = M.BatchNorm2d(w.shape[0], eps=BN_EPS)
            for a, v in ((bn.gamma.data, gamma), (bn.beta.data, beta), (bn.running_mean, mean),
                         (bn.running_var, var)):
                a[...] = v.double().cpu().numpy().reshape(a.shape)
            blocks.append(M.fuse(layer, bn, M.ReLU(), out_dtype="bf16"))
        head = M.Linear(case["c2"], LOGITS)
        head.weight = M.QuantizedParameters.from_float(t["w3"], "e4m3")
        head.bias = M.Parameters(t["b3"])
        s["net"] = (blocks[0], M.MaxPool2d(2, 2), blocks[1], M.GlobalAvgPool2d(), head)
    return s


def run(s):
    op, case = s["op"], s["case"]
    if op == "linear":
        y = F.linear(s["x"], s["weight"], s["bias"])
        if not case["train"]:
            return y
        return (y,) + F.linear_backward(s["g"], s["x"], s["weight"], case["bias"])
    if op == "conv":
        geometry = (case["k"], case["s"], case["p"])
        if case["fused"]:
            return F.conv2d(s["x"], s["weight"], *geometry, bias=s["bias"],
                            epilogue=s["epilogue"])
        y = F.conv2d(s["x"], s["weight"], *geometry, bias=s["bias"])
        if not case["train"]:
            return y
        return (y,) + F.conv2d_backward(s["g"], s["x"], s["weight"], *geometry)
    if op == "quantize":
        q = quant.quantize(s["x"], case["dtype"])
        return q.data.view(torch.uint8), q.scale, q.amax, quant.dequantize(q)
    if op == "maxpool":
        return s["layer"](s["x"]), s["layer"].backward(s["g"])
    if op == "adamw":
        w = s["weight"]
        w.grad = s["g"]
        s["opt"].step()
        return (w.codes.view(torch.uint8), w.scale, w.master, s["opt"].m_t[0], s["opt"].v_t[0])
    first, pool, second, gap, head = s["net"]
    features = second(pool(first(s["x"])))
    return features, head(gap(features).reshape(case["n"], -1))


# --------------------------------------------------------------------------
# what a pass cannot do without

_BYTES = {"f32": 4.0, "bf16": 2.0, "e4m3": 1.0, "e5m2": 1.0, "e2m1": 0.5}


def work(case):
    op = case["op"]
    if op == "linear":
        m, k, n = case["rows"], case["din"], case["dout"]
        b = m * k * _BYTES[case["xdtype"]] + n * k * _BYTES[case["wdtype"]] + 4 * m * n
        b += 4 * n if case["bias"] else 0
        if case["train"]:  # grad read; grad_input, grad_weight, grad_bias written
            b += 4 * (m * n + m * k + n * k) + (4 * n if case["bias"] else 0)
        return {"bytes": b, "flops": 2 * m * k * n * (3 if case["train"] else 1)}
    if op == "conv":
        oh, ow = _out(case)
        x, y = case["n"] * case["c"] * case["h"] * case["w"], case["n"] * case["co"] * oh * ow
        k = case["c"] * case["k"] * case["k"]
        w = case["co"] * k
        out = _BYTES[case["xdtype"]] if case["fused"] else 4
        b = x * _BYTES[case["xdtype"]] + w * _BYTES[case["wdtype"]] + y * out + 4 * case["co"]
        if case["fused"]:
            b += 8 * case["co"]
        if case["train"]:
            b += 4 * (y + x + w + case["co"])
        return {"bytes": b, "flops": 2 * y * k * (3 if case["train"] else 1)}
    if op == "quantize":  # x read, codes written and read, the fp32 values written
        n = case["n"]
        return {"bytes": n * (_BYTES[case["src"]] + 2 * _BYTES[case["dtype"]] + 4), "flops": 3 * n}
    if op == "maxpool":
        oh, ow = _out(case)
        x, y = (case["n"] * case["c"] * v for v in (case["h"] * case["w"], oh * ow))
        return {"bytes": x * (_BYTES[case["x"]] + 4) + y * (_BYTES[case["x"]] + 4),
                "flops": 2 * y * case["k"] ** 2}
    if op == "adamw":  # w, m, v read and written, the gradient read, codes written
        n = case["dout"] * case["din"]
        return {"bytes": n * (28 + _BYTES[case["dtype"]]), "flops": 15 * n}
    n, h, w, c1, c2 = (case[k] for k in ("n", "h", "w", "c1", "c2"))
    q = h // 4 * (w // 4)
    weights = (9 * c1 + 9 * c1 * c2) * _BYTES[case["dtype"]] + LOGITS * (c2 + 4)
    return {"bytes": 4 * n * h * w + 2 * n * c2 * q + 4 * n * LOGITS + weights + 16 * (c1 + c2),
            "flops": 2 * n * (9 * c1 * h * w + 9 * c1 * c2 * q + c2 * LOGITS)}


# --------------------------------------------------------------------------
# the same in 64 bits

def tolerance(case):
    """Products round their fp32 operands to bf16 (2^-9 at most, about 1.6e-3
    to 2.4e-3 over a result whose operand was fp32); bf16 outputs add as much
    again, and the CNN three such layers.  Operands that are bf16 already are
    multiplied exactly and summed in fp32.  Everything else is exact."""
    op = case["op"]
    if op == "linear":
        return {"rel": 8e-3 if case["xdtype"] == "f32" else 1e-5}
    if op == "conv":
        return {"rel": 8e-3 if case["xdtype"] == "f32" or case["fused"] else 1e-5}
    if op == "cnn":
        return {"rel": 1.5e-2}
    return "exact"


_FMT_MAX = {"e4m3": 448.0, "e5m2": 57344.0, "e2m1": 6.0}


def _quantized(w, dtype):
    """s * dec(codes) of w in 64 bits, and the fp32 scale s: s = amax / largest
    value, the code of w * (1 / s) rounded to nearest even."""
    # fp32 quotients, correctly rounded: the 64-bit ones rounded once more
    s = (w.abs().max().double() / _FMT_MAX[dtype]).float()
    v = (w.float() * (1.0 / s.double()).float()).clamp(-_FMT_MAX[dtype], _FMT_MAX[dtype])
    if dtype == "e2m1":
        a = v.abs()
        m = torch.zeros_like(a)
        # (bound, value at or above it, whether a tie goes up to the even code)
        for bound, value, up in ((0.25, 0.5, False), (0.75, 1.0, True), (1.25, 1.5, False),
                                 (1.75, 2.0, True), (2.5, 3.0, False), (3.5, 4.0, True),
                                 (5.0, 6.0, False)):
            m = torch.where(a >= bound if up else a > bound, torch.full_like(a, value), m)
        q = torch.copysign(m, v).double()
    else:
        q = v.to(torch.float8_e4m3fn if dtype == "e4m3" else torch.float8_e5m2).double()
    return q * s.double(), s


def _fold(gamma, beta, mean, var):
    mul = gamma.double() / torch.sqrt(var.double() + BN_EPS)
    return mul, beta.double() - mean.double() * mul


def _columns(x, k, s, p):
    """(C*k*k, N*OH*OW) window matrix of a float64 image batch, zero padding."""
    c = torch.nn.functional.unfold(x, k, padding=p, stride=s)
    return c.permute(1, 0, 2).reshape(c.shape[1], -1)


def _conv64(x, w, k, s, p):
    n, co = x.shape[0], w.shape[0]
    oh, ow = (x.shape[2] + 2 * p - k) // s + 1, (x.shape[3] + 2 * p - k) // s + 1
    y = w.reshape(co, -1) @ _columns(x, k, s, p)
    return y.reshape(co, n, oh, ow).permute(1, 0, 2, 3).contiguous()


def exact(case, seed):
    t, op = draws(case, seed), case["op"]
    if op == "linear":
        w, _ = _quantized(t["w"], case["wdtype"])
        x = t["x"].double()
        y = x @ w.T
        if case["bias"]:
            y = y + t["b"].double()
        if not case["train"]:
            return y
        g = t["g"].double()
        return y, g @ w, g.T @ x, g.sum(0, keepdim=True) if case["bias"] else None
    if op == "conv":
        k, s, p = case["k"], case["s"], case["p"]
        w, _ = _quantized(t["w"], case["wdtype"])
        x = t["x"].double()
        y = _conv64(x, w, k, s, p) + t["b"].double().reshape(1, -1, 1, 1)
        if case["fused"]:
            mul, add = _fold(t["gamma"], t["beta"], t["mean"], t["var"])
            y = (y * mul.reshape(1, -1, 1, 1) + add.reshape(1, -1, 1, 1)).relu()
        if not case["train"]:
            return y
        co, n = case["co"], case["n"]
        g = t["g"].double()
        flat = g.permute(1, 0, 2, 3).reshape(co, -1)
        gw = (flat @ _columns(x, k, s, p).T).reshape(w.shape)
        cols = (w.reshape(co, -1).T @ flat).reshape(-1, n, flat.shape[1] // n)
        gi = torch.nn.functional.fold(cols.permute(1, 0, 2).contiguous(),
                                      (case["h"], case["w"]), k, padding=p, stride=s)
        return y, gi, gw, g.sum((0, 2, 3)).reshape(co, 1)
    if op == "quantize":
        amax = t["x"].abs().max().double()
        return None, (amax / _FMT_MAX[case["dtype"]]).reshape(1), amax.reshape(1), None
    if op == "maxpool":
        k, s, p = case["k"], case["s"], case["p"]
        # the zero border takes part in the maximum, and in its ties; a
        # window's gradient is shared over the elements equal to its maximum
        n, c, h, w = t["x"].shape
        oh, ow = _out(case)
        x = t["x"].double().reshape(n * c, 1, h, w)
        cols = torch.nn.functional.unfold(x, k, padding=p, stride=s)
        top = cols.amax(1, keepdim=True)
        hit = (cols == top).double()
        share = hit * (t["g"].double().reshape(n * c, 1, -1) / hit.sum(1, keepdim=True))
        gi = torch.nn.functional.fold(share, (h, w), k, padding=p, stride=s)
        return top.reshape(n, c, oh, ow), gi.reshape(n, c, h, w)
    if op == "adamw":
        w, g = t["w"].double(), t["g"].double()
        b1, b2 = ADAM["betas"]
        m, v = (1 - b1) * g, (1 - b2) * g * g
        w = w - ADAM["lr"] * (m / (1 - b1)) / ((v / (1 - b2)).sqrt() + 1e-8)
        w = w - ADAM["lr"] * ADAM["weight_decay"] * w
        scale = (w.abs().max() / _FMT_MAX[case["dtype"]]).reshape(1)
        if case["dtype"] == "e2m1" and case["din"] % 2:  # stored in whole bytes a row
            w, m, v = (torch.nn.functional.pad(a, (0, 1)) for a in (w, m, v))
        return None, scale, w, m, v
    a = t["x"].double()
    for w, bn, stride in ((t["w1"], t["bn1"], 1), (t["w2"], t["bn2"], 2)):
        if stride == 2:
            a = torch.nn.functional.max_pool2d(a, 2)
        mul, add = _fold(*bn)
        y = _conv64(a, _quantized(w, case["dtype"])[0], 3, stride, 1)
        a = (y * mul.reshape(1, -1, 1, 1) + add.reshape(1, -1, 1, 1)).relu()
    w, _ = _quantized(t["w3"], "e4m3")
    return a, a.mean((2, 3)) @ w.T + t["b3"].double()
