"""Workloads of the PAM operators as a training or inference program runs them: what is timed when a kernel or its
host path changes.

Every case goes through the package's public entry points (`import pam_amd as pam`) with operands resident on the GPU.
`listed()` gives fixed cases, `draw(rng)` more of the same ranges, `prepare` the tensors a program holds before the call,
`run` one pass (forward, and the gradients where the case trains), `work` the bytes and lane-operations the pass cannot do
without and `tolerance` how far another correct order of the float32 sums may move the results.

Kinds:
  linear       pam.linear on [tokens, d_in]: the projections and feed-forward layers of a transformer, with or without bias,
               activations dense or after a ReLU (half zeros), the recipes' approximate gradients or the default exact ones
  attention    the core of an attention layer: pam.bmm (Q K^T), the causal mask, pam.softmax, pam.bmm (P V)
  layer_norm   pam.layer_norm over token rows
  log_softmax  pam.log_softmax over vocabulary rows with the gradient of a label-smoothed cross entropy
  elementwise  pam.mul / div / exp / log / pow over whole tensors
  conv         pam.conv2d / conv2d_group: 3 x 3 convolutions, patch embeddings, depthwise convolutions
  adam         one pam Adam step over all parameters of an encoder-decoder transformer
"""
import math

import torch

import pam_amd as pam
from pam_amd.optim import Adam

OFFSET = 1.0552            # the multiplier of the recipes that correct PAM's mean error


# ---------------------------------------------------------------- the cases

def _linear(tokens, d_in, d_out, approx=True, relu=False, bias=True, offset=False, train=True):
    return dict(kind="linear", tokens=tokens, d_in=d_in, d_out=d_out, approx=approx, relu=relu, bias=bias, offset=offset, train=train)


def _attention(heads, tq, tk, dh, causal=False, train=True):
    return dict(kind="attention", heads=heads, tq=tq, tk=tk, dh=dh, causal=causal, train=train)


def _conv(batch, c, side, co, kernel, stride, pad, groups=1, approx=True, input_grad=True):
    return dict(kind="conv", batch=batch, c=c, side=side, co=co, kernel=kernel, stride=stride, pad=pad, groups=groups, approx=approx,
                input_grad=input_grad)


def listed():
    def named(name, case):
        return dict(case, name=name)
    return [
        # the smallest training call: a layer of a 64-wide model on a batch of 8 x 12 tokens, all launches and host work
        named("linear_small", _linear(96, 64, 128)),
        # the first layer of the MLP of DeiT-tiny on 64 images of 197 tokens
        named("linear_deit_tiny", _linear(12608, 192, 768)),
        # a feed-forward layer of the translation model (4096 tokens per batch) with the default, exact gradients
        named("linear_exact", _linear(4096, 512, 1024, approx=False)),
        # the layer behind the ReLU of that feed-forward block: half of its input is zero
        named("linear_relu_input", _linear(4096, 1024, 512, relu=True, offset=True)),
        # the tied output projection onto a vocabulary of 10 000 words: the largest product
        named("linear_vocabulary", _linear(4096, 512, 10000, bias=False)),
        # attention of DeiT-tiny: 64 images x 3 heads, 197 tokens, 64 channels per head
        named("attention_deit_tiny", _attention(192, 197, 197, 64)),
        # one decoding step of the translation model's inference: one query token per sentence against 120 cached ones
        named("attention_decode", _attention(256, 1, 120, 64, train=False)),
        # the layer norms of DeiT-tiny on 256 images
        named("layer_norm_deit_tiny", dict(kind="layer_norm", rows=50432, width=192, approx=True)),
        # the loss of the translation model: 4096 tokens over the vocabulary, default gradients
        named("log_softmax_vocabulary", dict(kind="log_softmax", rows=4096, width=10000, approx=False)),
        # an elementwise product of large activations and both of its gradients
        named("elementwise_mul_large", dict(kind="elementwise", op="mul", n=1 << 26, approx=False, offset=False)),
        # a convolution of a small residual network
        named("conv_3x3", _conv(128, 64, 32, 128, 3, 1, 1)),
        # the optimizer step of the translation model: 253 tensors, 6 + 6 layers of width 512, feed-forward 1024
        named("adam_transformer", dict(kind="adam", width=512, ffn=1024, layers=6, vocabulary=10000)),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, evenly spread over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "attention", "attention", "layer_norm", "log_softmax", "elementwise", "conv", "adam"])
    approx = rng.random() < 0.6
    if kind == "linear":
        if rng.random() < 0.2:                     # inference on a few tokens
            return _linear(_spread(rng, 1, 512), _spread(rng, 48, 1024), _spread(rng, 48, 4096), train=False, bias=rng.random() < 0.7)
        d_in, d_out = _spread(rng, 48, 1024), _spread(rng, 48, 4096)
        if rng.random() < 0.6:                     # most models' widths are multiples of 32
            d_in, d_out = max(64, d_in // 32 * 32), max(64, d_out // 32 * 32)
        most = 20_000_000_000 // (d_in * d_out)
        return _linear(_spread(rng, 64, min(16384, most)), d_in, d_out, approx=approx, relu=rng.random() < 0.3, bias=rng.random() < 0.7,
                       offset=rng.random() < 0.2)
    if kind == "attention":
        dh = rng.choice([32, 48, 64, 64, 64, 80, 128])
        if rng.random() < 0.25:
            return _attention(_spread(rng, 8, 512), _spread(rng, 1, 4), _spread(rng, 8, 512), dh, train=False)
        t = _spread(rng, 16, 400)
        causal = rng.random() < 0.3
        tk = t if causal or rng.random() < 0.6 else _spread(rng, 16, 400)
        # approximate gradients, as every recipe has them: the exact ones of this chain jump with the last bit of a score,
        # and no two orders of the sums agree on them
        return _attention(_spread(rng, 8, max(8, min(256, 10_000_000 // (t * tk)))), t, tk, dh, causal=causal)
    if kind == "layer_norm":
        width = _spread(rng, 64, 1024)
        if rng.random() < 0.6:
            width = max(64, width // 32 * 32)
        return dict(kind="layer_norm", rows=_spread(rng, 64, min(65536, 40_000_000 // width)), width=width, approx=approx)
    if kind == "log_softmax":
        width = _spread(rng, 100, 32768)
        return dict(kind="log_softmax", rows=_spread(rng, 64, min(8192, 40_000_000 // width)), width=width, approx=approx)
    if kind == "elementwise":
        return dict(kind="elementwise", op=rng.choice(["mul", "div", "exp", "log", "pow"]), n=_spread(rng, 1000, 1 << 26), approx=approx,
                    offset=rng.random() < 0.2)
    if kind == "conv":
        which = rng.choice(["3x3", "3x3", "patches", "depthwise"])
        if which == "3x3":
            c, co, side = rng.choice([16, 32, 64, 96]), rng.choice([32, 64, 128]), rng.randint(8, 32)
            return _conv(_spread(rng, 4, 128), c, side, co, 3, 1, 1, approx=approx)
        if which == "patches":
            p = rng.choice([4, 8, 16])
            return _conv(_spread(rng, 4, 64), 3, p * rng.randint(7, 14), rng.choice([96, 192, 384]), p, p, 0, approx=approx, input_grad=False)
        c = rng.choice([32, 64, 96, 192])
        kernel = rng.choice([3, 5, 7])
        return _conv(_spread(rng, 4, 32), c, rng.randint(14, 28), c, kernel, 1, kernel // 2, groups=c, approx=approx)
    return dict(kind="adam", width=64 * rng.randint(1, 8), ffn=128 * rng.randint(1, 8), layers=rng.randint(1, 6), vocabulary=_spread(rng, 100, 10000))


# ---------------------------------------------------------------- the tensors a program holds before the call

def _maker(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * std
    return normal, g


def _leaf(t, train):
    return t.requires_grad_(True) if train else t


def _adam_shapes(case):
    w, f = case["width"], case["ffn"]
    attention = [(w, w), (w,)] * 4
    ffn = [(f, w), (f,), (w, f), (w,)]
    norm = [(w,), (w,)]
    encoder = attention + norm + ffn + norm
    decoder = attention + norm + attention + norm + ffn + norm
    return [(case["vocabulary"], w)] + case["layers"] * encoder + case["layers"] * decoder


def prepare(case, seed):
    normal, g = _maker(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "linear":
        t, i, o, train = case["tokens"], case["d_in"], case["d_out"], case["train"]
        x = normal(t, i)
        s["x"] = _leaf(x.relu_() if case["relu"] else x, train)
        s["w"] = _leaf(torch.nn.init.trunc_normal_(torch.empty(o, i, device="cuda"), std=0.02, a=-0.04, b=0.04, generator=g), train)
        s["b"] = _leaf(normal(o, std=0.02), train) if case["bias"] else None
        s["dy"] = normal(t, o, std=1e-2) if train else None
        s["kw"] = dict(offset=OFFSET if case["offset"] else None, approx_bwd=case["approx"])
    elif kind == "attention":
        h, tq, tk, dh, train = case["heads"], case["tq"], case["tk"], case["dh"], case["train"]
        s["q"] = _leaf(normal(h, tq, dh, std=dh ** -0.5), train)
        s["k"], s["v"] = _leaf(normal(h, tk, dh), train), _leaf(normal(h, tk, dh), train)
        s["mask"] = torch.ones(tq, tk, dtype=torch.bool, device="cuda").triu(1) if case["causal"] else None
        s["do"] = normal(h, tq, dh, std=1e-2) if train else None
        s["kw"] = dict(approx_bwd=True)
    elif kind == "layer_norm":
        s["x"] = normal(case["rows"], case["width"]).requires_grad_(True)
        s["w"] = normal(case["width"], std=0.1).add_(1.0).requires_grad_(True)
        s["b"] = normal(case["width"], std=0.1).requires_grad_(True)
        s["dy"] = normal(case["rows"], case["width"], std=1e-2)
    elif kind == "log_softmax":
        rows, n = case["rows"], case["width"]
        s["x"] = normal(rows, n, std=2.0).requires_grad_(True)
        dy = torch.full((rows, n), -0.1 / n / rows, device="cuda")
        dy[torch.arange(rows, device="cuda"), torch.randint(0, n, (rows,), generator=g, device="cuda")] -= 0.9 / rows
        s["dy"] = dy
    elif kind == "elementwise":
        a = normal(case["n"])
        s["a"] = (a.abs_().add_(1e-3) if case["op"] in ("log", "pow") else a).requires_grad_(True)
        s["b"] = normal(case["n"]).requires_grad_(True) if case["op"] in ("mul", "div") else None
        s["dy"] = normal(case["n"], std=1e-2)
        s["kw"] = dict(offset=OFFSET if case["offset"] else None, approx_bwd=case["approx"])
    elif kind == "conv":
        b, c, side, co, k = case["batch"], case["c"], case["side"], case["co"], case["kernel"]
        s["x"] = _leaf(normal(b, c, side, side), case["input_grad"])
        s["w"] = normal(co, c // case["groups"], k, k, std=(c // case["groups"] * k * k) ** -0.5).requires_grad_(True)
        s["b"] = normal(co, std=0.1).requires_grad_(True)
        out = (side + 2 * case["pad"] - k) // case["stride"] + 1
        s["dy"] = normal(b, co, out, out, std=1e-2)
    else:
        # a program in the middle of training: every parameter has its moments, kept in flat buffers as a checkpoint restores them
        shapes = _adam_shapes(case)
        sizes = [(math.prod(shape) + 63) // 64 * 64 for shape in shapes]
        total = sum(sizes)
        flat = {"p": normal(total, std=0.05), "g": normal(total, std=1e-3), "m": normal(total, std=1e-3), "v": normal(total, std=1e-3).square_()}
        params, at = [], 0
        for shape, size in zip(shapes, sizes):
            n = math.prod(shape)
            view = {key: buffer[at:at + n].view(shape) for key, buffer in flat.items()}
            p = torch.nn.Parameter(view["p"])
            p.grad = view["g"]
            params.append((p, view))
            at += size
        s["optimizer"] = Adam([p for p, _ in params], lr=5e-4, betas=(0.9, 0.98), eps=1e-8, weight_decay=1e-4, opt_functional_cfg="pam")
        for p, view in params:
            s["optimizer"].state[p] = {"step": 1000, "exp_avg": view["m"], "exp_avg_sq": view["v"]}
        s["flat"] = flat
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        y = pam.linear(s["x"], s["w"], s["b"], **s["kw"])
        if not case["train"]:
            return y
        return y, torch.autograd.grad(y, [t for t in (s["x"], s["w"], s["b"]) if t is not None], s["dy"])
    if kind == "attention":
        scores = pam.bmm(s["q"], s["k"].transpose(1, 2), **s["kw"])
        if s["mask"] is not None:
            scores = scores.masked_fill(s["mask"], float("-inf"))
        y = pam.bmm(pam.softmax(scores, dim=-1, **s["kw"]), s["v"], **s["kw"])
        if not case["train"]:
            return y
        return y, torch.autograd.grad(y, (s["q"], s["k"], s["v"]), s["do"])
    if kind == "layer_norm":
        y = pam.layer_norm(s["x"], case["width"], s["w"], s["b"], approx_bwd=case["approx"])
        return y, torch.autograd.grad(y, (s["x"], s["w"], s["b"]), s["dy"])
    if kind == "log_softmax":
        y = pam.log_softmax(s["x"], dim=-1, approx_bwd=case["approx"])
        return y, torch.autograd.grad(y, s["x"], s["dy"])
    if kind == "elementwise":
        op = case["op"]
        if op in ("mul", "div"):
            y = getattr(pam, op)(s["a"], s["b"], **s["kw"])
            return y, torch.autograd.grad(y, (s["a"], s["b"]), s["dy"])
        y = pam.pow(s["a"], 0.5, **s["kw"]) if op == "pow" else getattr(pam, op)(s["a"], **s["kw"])
        return y, torch.autograd.grad(y, s["a"], s["dy"])
    if kind == "conv":
        kw = dict(stride=case["stride"], padding=case["pad"], approx_bwd=case["approx"])
        if case["groups"] > 1:
            y = pam.conv2d_group(s["x"], s["w"], s["b"], groups=case["groups"], **kw)
        else:
            y = pam.conv2d(s["x"], s["w"], s["b"], **kw)
        return y, torch.autograd.grad(y, ([s["x"]] if case["input_grad"] else []) + [s["w"], s["b"]], s["dy"])
    s["optimizer"].step()
    return s["flat"]["p"], s["flat"]["m"], s["flat"]["v"]


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Bytes: every input read once, every output written once, float32.  Operations: two lane-operations per PAM
    multiply-accumulate (an integer and a float add), three in an exact gradient; a few per element elsewhere."""
    kind = case["kind"]
    if kind == "linear":
        t, i, o = case["tokens"], case["d_in"], case["d_out"]
        bias = o if case["bias"] else 0
        macs = t * i * o
        if not case["train"]:
            return {"bytes": 4 * (t * i + i * o + bias + t * o), "flops": 2 * macs}
        # x, w, b, dy in; y, dx, dw, db out
        return {"bytes": 4 * 2 * (t * i + i * o + bias + t * o), "flops": (2 + 2 * (2 if case["approx"] else 3)) * macs}
    if kind == "attention":
        h, tq, tk, dh = case["heads"], case["tq"], case["tk"], case["dh"]
        macs, ends, scores = h * tq * tk * dh, h * (2 * tq + 2 * tk) * dh, h * tq * tk
        if not case["train"]:
            return {"bytes": 4 * (ends + 4 * scores), "flops": 4 * macs}
        # q, k, v, do in; y, dq, dk, dv out; the scores and the weights and their gradients go out and come in again
        return {"bytes": 4 * (2 * ends + 10 * scores), "flops": 12 * macs}
    if kind == "layer_norm":
        n = case["rows"] * case["width"]
        return {"bytes": 4 * (5 * n + 5 * case["width"]), "flops": 30 * n}      # x, y; x, dy, dx
    if kind == "log_softmax":
        n = case["rows"] * case["width"]
        return {"bytes": 4 * 6 * n, "flops": 30 * n}                            # x (for the maximum of all), x, y; x, dy, dx
    if kind == "elementwise":
        return {"bytes": 4 * case["n"] * (8 if case["op"] in ("mul", "div") else 5), "flops": 10 * case["n"]}
    if kind == "conv":
        out = (case["side"] + 2 * case["pad"] - case["kernel"]) // case["stride"] + 1
        x = case["batch"] * case["c"] * case["side"] ** 2
        y = case["batch"] * case["co"] * out * out
        per = case["c"] // case["groups"] * case["kernel"] ** 2
        ops = 2 + (2 if case["approx"] else 3) * (2 if case["input_grad"] else 1)
        return {"bytes": 4 * (x * (3 if case["input_grad"] else 2) + 2 * y + 3 * case["co"] * per), "flops": ops * y * per}
    n = sum(math.prod(shape) for shape in _adam_shapes(case))
    return {"bytes": 28 * n, "flops": 30 * n}


def tolerance(case):
    """How far the results move when the terms of the float32 sums are added in another order: measured by permuting the
    summed dimensions of the inputs, times about four.  The exact gradient of layer_norm has steps (a slope is a power of
    two that jumps where a mantissa sum carries), and behind a row's sum a few of its values move by half their size."""
    kind = case["kind"]
    if kind in ("elementwise", "adam"):
        return "exact"                             # no sums: every operation is defined to the bit
    if kind == "linear":
        return {"rel": 8e-6}
    if kind == "conv":
        return {"rel": 4e-6}
    if kind == "attention":
        return {"rel": 3e-6}
    if kind == "layer_norm" and not case["approx"]:
        return {"rel": 2.5e-3, "max": 0.99}
    return {"rel": 1e-6, "max": 1e-4}
