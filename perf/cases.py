"""What the library's speed is judged by: the work its users have it do, through its public entry points, over the
range of sizes, layouts and types they meet.

Every case names a `path` (one of the programs below) and its sizes.  Operands are made on the GPU from the seed;
outputs are written to buffers the state owns, as a program that calls the device entry points in a loop keeps them.
The two paths on host data (`host_gemm`, `classifier`) take numpy arrays through the whole call, copies included.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from spiraltorch_amd import hip
from spiraltorch_amd.tensor import Linear, Tensor

RELU, GELU = int(hip.GemmActivation.Relu), int(hip.GemmActivation.Gelu)


def listed():
    return [
        # The drop-in call of the backend crate on host slices (relu(A.B + bias), operands copied in, result copied
        # out), at the smallest size of the benchmark: what a program that keeps its tensors on the host pays.
        {"name": "host_gemm_512", "path": "host_gemm", "m": 512, "n": 512, "k": 512},
        # A classifier called on a host batch through the operator mirror: two Linear layers with a GELU between, row
        # softmax, probabilities back on the host.  A chain of small calls: launches, checks and allocations count.
        {"name": "classifier_64", "path": "classifier", "rows": 64, "inputs": 784, "hidden": 512, "classes": 1000},
        # Training step (forward and all gradients) of a vision transformer's MLP block on 8 images of 197 tokens:
        # every f32 GEMM layout (row-major, A transposed, B prepacked), column sums, GELU and its derivative.
        {"name": "mlp_step_1576", "path": "mlp_step", "tokens": 1576, "width": 768, "hidden": 3072},
        # Training step of a 3x3 convolution layer: forward and the three gradients (the benchmark's layer).
        {"name": "conv_step_56", "path": "conv_step", "batch": 32, "c_in": 64, "c_out": 128, "h": 56, "w": 56,
         "kernel": 3, "stride": 1, "padding": 1},
        # Inference through a deep layer of a residual network on bf16 activations.
        {"name": "conv_bf16_14", "path": "conv_bf16", "batch": 32, "c_in": 256, "c_out": 256, "h": 14, "w": 14,
         "kernel": 3, "stride": 1, "padding": 1},
        # Causal self-attention in f32: 8 sequences of 2048 tokens, 16 heads.
        {"name": "attention_causal_2048", "path": "attention", "contexts": 128, "sequence": 2048, "head_dim": 64,
         "causal": True, "biased": False},
        # Attention within one context under a per-key and a per-pair bias: the reference's own use of the operator.
        {"name": "attention_biased_1000", "path": "attention", "contexts": 1, "sequence": 1000, "head_dim": 64,
         "causal": False, "biased": True},
        # The benchmark's large bf16 product, both operands row-major, f32 out.
        {"name": "gemm_bf16_4096", "path": "gemm_bf16", "m": 4096, "n": 4096, "k": 4096, "packed": False,
         "activation": 0, "out_bf16": False},
        # A decode step's projection: 16 rows against a prepacked 4096 x 4096 weight, with bias.
        {"name": "gemm_bf16_16_rows", "path": "gemm_bf16", "m": 16, "n": 4096, "k": 4096, "packed": True,
         "activation": 0, "out_bf16": False},
        # A language-model head over a vocabulary that is no multiple of anything, and its softmax.
        {"name": "lm_head_50257", "path": "lm_head", "rows": 1024, "width": 768, "vocab": 50257},
        # The byte-level decoder on one short prompt (latency) ...
        {"name": "decoder_1x117", "path": "decoder", "batch": 1, "seq": 117, "width": 512, "heads": 8, "layers": 6},
        # ... and on the benchmark's batch (throughput).
        {"name": "decoder_16x1024", "path": "decoder", "batch": 16, "seq": 1024, "width": 512, "heads": 8, "layers": 6},
    ]


def _log(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _size(rng, low, high):
    """Log-uniform over low..high; half the time the multiple of 64 (16 below 64) nearby, as widths usually are, and as
    it fell, odd sizes among them, otherwise."""
    value = _log(rng, low, high)
    step = 64 if value >= 64 else 16
    if rng.random() < 0.5 and value > step // 2:
        value = min(high, max(low, (value + step // 2) // step * step))
    return value


def draw(rng):
    path = rng.choice(["host_gemm", "classifier", "mlp_step", "conv_step", "conv_bf16", "attention", "gemm_bf16",
                       "lm_head", "decoder"])
    while True:
        case = {"path": path}
        if path == "host_gemm":
            case.update(m=_size(rng, 16, 1024), n=_size(rng, 16, 1024), k=_size(rng, 16, 1024))
        elif path == "classifier":
            case.update(rows=_size(rng, 1, 2048), inputs=_size(rng, 16, 1024), hidden=_size(rng, 16, 1024),
                        classes=_size(rng, 2, 1024))
        elif path == "mlp_step":
            width = _size(rng, 32, 1024)
            case.update(tokens=_size(rng, 8, 4096), width=width, hidden=rng.choice([2, 3, 4]) * width)
        elif path in ("conv_step", "conv_bf16"):
            kernel = rng.choice([1, 3, 3, 3, 5, 7])
            stride = rng.choice([1, 1, 1, 2])
            side = _log(rng, 7, 112)
            case.update(batch=_log(rng, 1, 32), c_in=rng.choice([3, 16, 24, 32, 64, 96, 128, 192, 256, 512]),
                        c_out=rng.choice([16, 32, 64, 96, 128, 192, 256, 512]), h=side, w=side + rng.choice([0, 0, 0, 1, 5]),
                        kernel=kernel, stride=stride, padding=kernel // 2)
        elif path == "attention":
            biased = rng.random() < 0.4
            case.update(contexts=_log(rng, 1, 16 if biased else 128), sequence=_size(rng, 16, 2048),
                        head_dim=rng.choice([32, 64, 64, 80, 128]), causal=not biased and rng.random() < 0.5, biased=biased)
        elif path == "gemm_bf16":
            case.update(m=_size(rng, 1, 8192), n=_size(rng, 256, 8192), k=_size(rng, 256, 8192), packed=rng.random() < 0.5,
                        activation=rng.choice([0, 0, RELU, GELU]), out_bf16=rng.random() < 0.5)
        elif path == "lm_head":
            case.update(rows=_size(rng, 1, 2048), width=rng.choice([256, 384, 512, 768, 1024]), vocab=_size(rng, 256, 50304))
        else:
            width, heads = rng.choice([(256, 4), (512, 8), (512, 4), (768, 12)])
            case.update(batch=_log(rng, 1, 16), seq=_log(rng, 1, 1024), width=width, heads=heads,
                        layers=rng.choice([2, 4, 6]))
        if _affordable(case):
            return case


# No drawn case asks for more than its path's largest listed one does.
_MOST = {"host_gemm": 2.2e9, "classifier": 4e9, "mlp_step": 45e9, "conv_step": 45e9, "conv_bf16": 45e9,
         "attention": 70e9, "gemm_bf16": 140e9, "lm_head": 110e9, "decoder": 730e9}


def _affordable(case):
    cost = work(case)
    return cost["flops"] <= _MOST[case["path"]] and cost["bytes"] <= 1.0e9


# ---- operands -----------------------------------------------------------------------------------------------------

class _Source:
    """Random operands on the GPU from one seed."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda")
        self.generator.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.generator, device="cuda") * std

    def uniform(self, *shape, bound=1.0):
        return (torch.rand(*shape, generator=self.generator, device="cuda") * 2.0 - 1.0) * bound

    def bf16(self, *shape, std=1.0):
        return self.normal(*shape, std=std).to(torch.bfloat16)


def _f32(*shape):
    return torch.empty(*shape, device="cuda")


def _conv_geometry(case):
    pair = lambda v: (v, v)
    return pair(case["kernel"]), pair(case["stride"]), pair(case["padding"]), (1, 1)


def _conv_output(case):
    side = lambda v: (v + 2 * case["padding"] - case["kernel"]) // case["stride"] + 1
    return side(case["h"]), side(case["w"])


VOCAB = 256  # byte-level decoder


def prepare(case, seed):
    src, path, s = _Source(seed), case["path"], {"case": case}
    if path == "host_gemm":
        m, n, k = case["m"], case["n"], case["k"]
        s.update(a=src.uniform(m, k).cpu().numpy(), b=src.uniform(k, n).cpu().numpy(), bias=src.uniform(n, bound=0.5).cpu().numpy(),
                 out=np.zeros(m * n, np.float32))
    elif path == "classifier":
        def layer(name, fan_in, fan_out):
            linear = Linear(name, fan_in, fan_out)
            linear.load_weight(Tensor.from_numpy(src.normal(fan_in, fan_out, std=math.sqrt(2.0 / fan_in)).cpu().numpy()),
                               Tensor.from_numpy(src.uniform(1, fan_out, bound=0.1).cpu().numpy()))
            return linear

        s.update(x=src.normal(case["rows"], case["inputs"]).cpu().numpy(), fc1=layer("fc1", case["inputs"], case["hidden"]),
                 fc2=layer("fc2", case["hidden"], case["classes"]))
    elif path == "mlp_step":
        t, d, f = case["tokens"], case["width"], case["hidden"]
        s.update(x=src.normal(t, d), g=src.normal(t, d), w1=src.normal(d, f, std=math.sqrt(2.0 / d)), b1=src.uniform(f, bound=0.1),
                 w2=src.normal(f, d, std=math.sqrt(1.0 / f)), b2=src.uniform(d, bound=0.1), z=_f32(t, f), h=_f32(t, f), y=_f32(t, d),
                 gh=_f32(t, f), gz=_f32(t, f), gx=_f32(t, d), gw1=_f32(d, f), gb1=_f32(f), gw2=_f32(f, d), gb2=_f32(d))
    elif path in ("conv_step", "conv_bf16"):
        n, ci, co, kk = case["batch"], case["c_in"], case["c_out"], case["kernel"]
        oh, ow = _conv_output(case)
        std = math.sqrt(2.0 / (ci * kk * kk))
        s.update(bias=src.uniform(co, bound=0.1))
        if path == "conv_bf16":
            s.update(x=src.bf16(n, ci, case["h"], case["w"]), w=src.bf16(co, ci, kk, kk, std=std),
                     y=torch.empty(n, co, oh, ow, device="cuda", dtype=torch.bfloat16))
        else:
            s.update(x=src.normal(n, ci, case["h"], case["w"]), w=src.normal(co, ci, kk, kk, std=std), g=src.normal(n, co, oh, ow),
                     y=_f32(n, co, oh, ow), gx=_f32(n, ci, case["h"], case["w"]), gw=_f32(co, ci, kk, kk), gb=_f32(co))
    elif path == "attention":
        c, n, d = case["contexts"], case["sequence"], case["head_dim"]
        s.update({name: src.normal(c, n, d) for name in "qkv"})
        s.update(out=_f32(c, n, d), z_bias=src.normal(c, n, std=0.5) if case["biased"] else None,
                 attn_bias=src.normal(c, n, n, std=0.5) if case["biased"] else None)
    elif path in ("gemm_bf16", "lm_head"):
        head = path == "lm_head"
        m, n, k = (case["rows"], case["vocab"], case["width"]) if head else (case["m"], case["n"], case["k"])
        packed = head or case["packed"]
        # N(0, 0.02^2) are the benchmark's operands; a head multiplies normalised activations.
        s.update(a=src.bf16(m, k, std=1.0 if head else 0.02), b=src.bf16(*((n, k) if packed else (k, n)), std=0.02),
                 bias=src.uniform(n, bound=0.1) if head or case["packed"] or case["activation"] else None)
        s.update(out=torch.empty(m, n, device="cuda", dtype=torch.bfloat16 if not head and case["out_bf16"] else torch.float32))
        if head:
            s.update(p=_f32(m, n))
    else:
        b, n, d, layers = case["batch"], case["seq"], case["width"], case["layers"]
        parts = [src.normal(VOCAB * d, std=0.02)]
        norm = [torch.ones(d, device="cuda"), torch.zeros(d, device="cuda")]
        for _ in range(layers):
            parts += norm + [src.normal(d * 3 * d + 3 * d + d * d + d, std=0.02)]
            parts += norm + [src.normal(d * 4 * d + 4 * d + 4 * d * d + d, std=0.02)]
        parts += norm + [src.normal(d * VOCAB + VOCAB, std=0.02)]
        weights = torch.cat(parts).cpu().numpy()
        s.update(decoder=hip.Decoder(VOCAB, d, case["heads"], layers, 4 * d, b, n, 1e-5, weights),
                 tokens=torch.randint(0, VOCAB, (b, n), generator=src.generator, device="cuda").float(), logits=_f32(b, n, VOCAB))
    return s


# ---- one pass -----------------------------------------------------------------------------------------------------

def _at(tensor):
    return None if tensor is None else tensor.data_ptr()


def run(s):
    case = s["case"]
    return _PATHS[case["path"]](case, s)


def _host_gemm(case, s):
    hip.gemm_bias_activation_f32(case["m"], case["n"], case["k"], hip.GemmActivation.Relu, s["a"], s["b"], s["bias"], None, s["out"])
    return s["out"]


def _classifier(case, s):
    hidden = s["fc1"].forward(Tensor.from_numpy(s["x"])).gelu()
    return s["fc2"].forward(hidden).row_softmax().numpy()


def _mlp_step(case, s):
    t, d, f = case["tokens"], case["width"], case["hidden"]
    p = {name: _at(value) for name, value in s.items() if name != "case"}
    hip.gemm_bias_act_f32_dev(t, f, d, 0, p["x"], p["w1"], p["b1"], None, p["z"])
    hip.gelu_f32_dev(t * f, p["z"], p["h"])
    hip.gemm_bias_act_f32_dev(t, d, f, 0, p["h"], p["w2"], p["b2"], None, p["y"])
    hip.gemm_f32_dev(f, d, t, 1.0 / t, True, p["h"], p["g"], p["gw2"])
    hip.sum_axis0_f32_dev(t, d, p["g"], 1.0 / t, p["gb2"])
    # a weight stored (in, out) is its own transpose in the prepacked layout
    hip.gemm_prepacked_bias_act_f32_dev(t, f, d, 0, p["g"], p["w2"], None, None, p["gh"])
    hip.gelu_backward_f32_dev(t * f, p["z"], p["gh"], p["gz"])
    hip.gemm_f32_dev(d, f, t, 1.0 / t, True, p["x"], p["gz"], p["gw1"])
    hip.sum_axis0_f32_dev(t, f, p["gz"], 1.0 / t, p["gb1"])
    hip.gemm_prepacked_bias_act_f32_dev(t, d, f, 0, p["gz"], p["w1"], None, None, p["gx"])
    return {name: s[name] for name in ("y", "gx", "gw1", "gb1", "gw2", "gb2")}


def _conv_step(case, s):
    shape = (case["batch"], case["c_in"], case["h"], case["w"], case["c_out"], *_conv_geometry(case))
    scale = 1.0 / case["batch"]
    hip.conv2d_bias_act_f32_dev(*shape, 0, _at(s["x"]), _at(s["w"]), _at(s["bias"]), _at(s["y"]))
    hip.conv2d_grad_weight_f32_dev(*shape, _at(s["x"]), _at(s["g"]), scale, _at(s["gw"]))
    hip.conv2d_grad_bias_f32_dev(*shape, _at(s["g"]), scale, _at(s["gb"]))
    hip.conv2d_grad_input_f32_dev(*shape, _at(s["g"]), _at(s["w"]), _at(s["gx"]))
    return {name: s[name] for name in ("y", "gx", "gw", "gb")}


def _conv_bf16(case, s):
    hip.conv2d_bias_act_bf16_dev(case["batch"], case["c_in"], case["h"], case["w"], case["c_out"], *_conv_geometry(case), RELU,
                                 _at(s["x"]), _at(s["w"]), _at(s["bias"]), None, _at(s["y"]))
    return s["y"]


def _attention(case, s):
    hip.attention_f32_dev(case["contexts"], case["sequence"], case["head_dim"], 1.0 / math.sqrt(case["head_dim"]), case["causal"],
                          _at(s["q"]), _at(s["k"]), _at(s["v"]), _at(s["z_bias"]), _at(s["attn_bias"]), _at(s["out"]))
    return s["out"]


def _gemm_bf16(case, s):
    call = hip.gemm_bf16_prepacked_bias_act_dev if case["packed"] else hip.gemm_bf16_bias_act_dev
    out = _at(s["out"])
    call(case["m"], case["n"], case["k"], case["activation"], _at(s["a"]), _at(s["b"]), _at(s["bias"]), None,
         None if case["out_bf16"] else out, out if case["out_bf16"] else None)
    return s["out"]


def _lm_head(case, s):
    m, n, k = case["rows"], case["vocab"], case["width"]
    hip.gemm_bf16_prepacked_bias_act_dev(m, n, k, 0, _at(s["a"]), _at(s["b"]), _at(s["bias"]), None, _at(s["out"]), None)
    hip.row_softmax_f32_dev(m, n, _at(s["out"]), _at(s["p"]))
    return {"logits": s["out"], "p": s["p"]}


def _decoder(case, s):
    s["decoder"].forward_dev(_at(s["tokens"]), _at(s["logits"]))
    return s["logits"]


_PATHS = {"host_gemm": _host_gemm, "classifier": _classifier, "mlp_step": _mlp_step, "conv_step": _conv_step, "conv_bf16": _conv_bf16,
          "attention": _attention, "gemm_bf16": _gemm_bf16, "lm_head": _lm_head, "decoder": _decoder}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def work(case):
    path = case["path"]
    if path == "host_gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + k * n + n + m * n), "flops": 2 * m * n * k}
    if path == "classifier":
        r, i, h, c = case["rows"], case["inputs"], case["hidden"], case["classes"]
        return {"bytes": 4 * (r * i + i * h + h + h * c + c + r * c), "flops": 2 * r * (i * h + h * c)}
    if path == "mlp_step":
        t, d, f = case["tokens"], case["width"], case["hidden"]
        return {"bytes": 4 * (4 * t * d + 4 * d * f + 2 * (d + f)), "flops": 12 * t * d * f}
    if path in ("conv_step", "conv_bf16"):
        n, ci, co, kk = case["batch"], case["c_in"], case["c_out"], case["kernel"]
        oh, ow = _conv_output(case)
        x, w, y = n * ci * case["h"] * case["w"], co * ci * kk * kk, n * co * oh * ow
        flops = 2 * y * ci * kk * kk
        if path == "conv_bf16":
            return {"bytes": 2 * (x + w + y) + 4 * co, "flops": flops}
        return {"bytes": 4 * (2 * x + 2 * w + 2 * y + 2 * co), "flops": 3 * flops}
    if path == "attention":
        c, n, d = case["contexts"], case["sequence"], case["head_dim"]
        pairs = n * (n + 1) // 2 if case["causal"] else n * n
        bias = c * n + c * n * n if case["biased"] else 0
        return {"bytes": 4 * (4 * c * n * d + bias), "flops": 4 * d * c * pairs}
    if path == "gemm_bf16":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + k * n) + (2 if case["out_bf16"] else 4) * m * n, "flops": 2 * m * n * k}
    if path == "lm_head":
        m, n, k = case["rows"], case["vocab"], case["width"]
        return {"bytes": 2 * (m * k + k * n) + 4 * n + 8 * m * n, "flops": 2 * m * n * k}
    t, d, layers = case["batch"] * case["seq"], case["width"], case["layers"]
    pairs = case["batch"] * (case["seq"] * (case["seq"] + 1) // 2)
    weights = layers * 12 * d * d + d * VOCAB
    return {"bytes": 2 * weights + 4 * t * (1 + VOCAB), "flops": 2 * t * weights + layers * 4 * d * pairs}


def tolerance(case):
    """About four times the largest error against float64 seen over the listed and some thirty drawn cases."""
    if case["path"] == "decoder":
        return {"rel": 1.5e-2, "max": 8e-2}  # bf16 operands through up to 6 layers: 0.3 to 0.5 % of the logits' rms
    if case["path"] == "conv_bf16" or (case["path"] == "gemm_bf16" and case["out_bf16"]):
        return {"rel": 7e-3, "max": 1.6e-2}  # seen 1.7e-3 and 3.9e-3: the rounding of the output to bf16
    if case["path"] in ("gemm_bf16", "lm_head"):
        return {"rel": 1.6e-6, "max": 1.4e-5}  # seen 4e-7 and 3.4e-6: exact products, f32 sums
    return {"rel": 8e-6, "max": 3.3e-5}  # seen 1.9e-6 and 8.2e-6: f32 throughout
