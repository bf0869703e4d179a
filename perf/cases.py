"""The work a program has torch_xdna do on one MI355X, as cases that can be timed and compared.

Each case goes through an op that the backend puts into a compiled graph (torch.ops.xdna.*), or, for
the attention layer of the Qwen3 stack, through its launcher. `prepare` makes what the program holds
before the call (tensors on the GPU from the seed, weights in the model's dtype, the options), `run`
is one call, `exact` the same values from plain torch in 64 bits.

Activations of linears are N(0, 1) with 0.1% outliers of 20 times that, weights N(0, 0.02), biases
N(0, 0.01); images N(0, 1); queries and keys what RMSNorm over a head leaves (unit variance).
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torch-xdna_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from torch_xdna import Config, kernels, ops, stack  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
ESZ = {"f32": 4, "bf16": 2, "f16": 2}
NH, NKV, DH, D, INTER = stack.NH, stack.NKV, stack.DH, stack.D, stack.INTER

# VGG-16's convs: output channels, "M" a 2x2 max-pool before the next conv
VGG16 = "64 64 M 128 128 M 256 256 256 M 512 512 512 M 512 512 512"


# ------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one token of one sequence through an attention projection: the smallest call, all latency
        {"name": "decode one row", "kind": "linear", "m": 1, "k": 4096, "parts": "4096", "dtype": "bf16", "bias": True,
         "precision": "int8"},
        # a decode step of 40 sequences through a wide MLP projection: bound by the weight stream
        {"name": "decode 40 rows", "kind": "linear", "m": 40, "k": 4096, "parts": "14336", "dtype": "bf16",
         "bias": True, "precision": "int8"},
        # q | k | v of a 699-token prompt as one GEMM: a short prefill with a ragged row count
        {"name": "qkv 699 rows", "kind": "linear", "m": 699, "k": 1024, "parts": "2048 1024 1024", "dtype": "bf16",
         "bias": False, "precision": "int8"},
        # the large prefill GEMM: the biggest W8A8 linear of the repository's configurations
        {"name": "prefill 8192 rows", "kind": "linear", "m": 8192, "k": 4096, "parts": "14336", "dtype": "bf16",
         "bias": True, "precision": "int8"},
        # a float32 model whose widths are no multiples of anything: rows without 16-byte alignment
        {"name": "odd sizes", "kind": "linear", "m": 1999, "k": 1537, "parts": "1001", "dtype": "f32", "bias": True,
         "precision": "int8"},
        # precision "bf16": the down projection of a float16 model at 512 rows
        {"name": "precision bf16", "kind": "linear", "m": 512, "k": 3072, "parts": "1024", "dtype": "f16",
         "bias": True, "precision": "bf16"},
        # one large 256-channel conv with its quantize and dequantize, as an unchained layer runs
        {"name": "conv 256 channels", "kind": "conv", "n": 1, "ci": 256, "co": 256, "h": 1536, "w": 64, "dtype": "f32",
         "bias": False, "relu": True},
        # a bf16 conv of odd channel counts on odd images, biased, signed outputs
        {"name": "conv ragged", "kind": "conv", "n": 4, "ci": 100, "co": 200, "h": 75, "w": 93, "dtype": "bf16",
         "bias": True, "relu": False},
        # four 256-channel convs with ReLU on a small image, kept int8 in between: a latency-bound chain
        {"name": "chain 64x64", "kind": "chain", "n": 1, "ci": 256, "layers": "256 256 256 256", "h": 64, "w": 64,
         "dtype": "f32", "bias": False},
        # VGG-16's 13 convs with their biases, ReLUs and pools at batch 8: a whole network's body
        {"name": "vgg-16 features", "kind": "chain", "n": 8, "ci": 3, "layers": VGG16, "h": 224, "w": 224,
         "dtype": "f32", "bias": True},
        # one attention layer over sequences of up to the longest length the stack takes
        {"name": "attention 4096", "kind": "attention", "lens": "4096 1500 700"},
        # the whole Qwen3-0.6B-width stack and head on two sequences (a long text's step)
        {"name": "qwen3 stack", "kind": "stack", "layers": 28, "out": 8200, "lens": "264 222"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """A size of [lo, hi], log-uniform: a multiple of `step` two times in three, else whatever it is."""
    v = _log(rng, lo, hi)
    return max(lo, min(hi, v // step * step if rng.random() < 0.67 else v))


MOST_MACS = 8192 * 4096 * 14336


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["conv"] * 3 + ["chain", "attention", "stack"])
    if kind == "linear":
        while True:
            m = rng.choice([1, _log(rng, 2, 64), _log(rng, 64, 8192), _log(rng, 64, 8192)])
            k, n = _size(rng, 256, 14336, 64), _size(rng, 256, 14336, 64)
            if m * k * n <= MOST_MACS // 2:
                break
        cut = rng.choice([1, 1, 2, 3])
        parts = [n // cut] * (cut - 1)
        parts.append(n - sum(parts))
        return {"kind": "linear", "m": m, "k": k, "parts": " ".join(map(str, parts)),
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "bias": rng.random() < 0.5,
                "precision": "bf16" if rng.random() < 0.2 else "int8"}
    if kind == "conv":
        while True:
            n, h, w = _log(rng, 1, 8), _size(rng, 14, 512, 8), _size(rng, 14, 256, 8)
            ci, co = rng.choice([3, _size(rng, 16, 512, 16)]), _size(rng, 16, 512, 16)
            if n * h * w * ci * co * 9 <= MOST_MACS // 4 and n * h * w * max(ci, co) <= 1 << 27:
                break
        bias = rng.random() < 0.5
        return {"kind": "conv", "n": n, "ci": ci, "co": co, "h": h, "w": w,
                "dtype": rng.choice(["f32", "bf16", "f16"]), "bias": bias, "relu": not bias}
    if kind == "chain":
        c = rng.choice([32, 48, 64, 96, 128, 256])
        layers = "%d %d M %d %d" % (c, c, 2 * c, 2 * c) if rng.random() < 0.5 else "%d %d %d" % (c, c, c)
        return {"kind": "chain", "n": _log(rng, 1, 4), "ci": rng.choice([3, c]), "layers": layers,
                "h": _size(rng, 28, 160, 4), "w": _size(rng, 28, 160, 4), "dtype": rng.choice(["f32", "bf16"]),
                "bias": rng.random() < 0.5}
    lens = [_log(rng, 20, 2500 if kind == "attention" else 700) for _ in range(rng.randint(1, 4))]
    if kind == "attention":
        return {"kind": "attention", "lens": " ".join(map(str, lens))}
    return {"kind": "stack", "layers": rng.choice([2, 4, 8]), "out": _size(rng, 256, 8200, 64),
            "lens": " ".join(map(str, lens))}


# ------------------------------------------------------------------------------ inputs
class _Rand:
    """Tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype="f32"):
        return (torch.randn(*shape, generator=self.g, device=self.dev) * std).to(DTYPES[dtype])

    def activations(self, m, k, dtype):
        x = torch.randn(m, k, generator=self.g, device=self.dev)
        far = torch.rand(m, k, generator=self.g, device=self.dev) < 1e-3
        return torch.where(far, 20 * x, x).to(DTYPES[dtype])

    def conv(self, co, ci, dtype):
        """A conv's default initialisation: uniform within 1 / sqrt(fan in)."""
        u = torch.rand(co, ci, 3, 3, generator=self.g, device=self.dev) * 2 - 1
        return (u / math.sqrt(9 * ci)).to(DTYPES[dtype])


def _parts(case):
    return [int(v) for v in case["parts"].split()]


def _lens(case):
    return [int(v) for v in case["lens"].split()]


def _chain(case):
    """(output channels, pool after this layer) of each layer."""
    out = []
    for v in case["layers"].split():
        if v == "M":
            out[-1] = (out[-1][0], True)
        else:
            out.append((int(v), False))
    return out


def _config(precision="int8"):
    return ops.config_id(Config(policy="gpu", verify="off", precision=precision))


def _linear_inputs(case, seed):
    r = _Rand(seed)
    dt = case["dtype"]
    x = r.activations(case["m"], case["k"], dt)
    ws = [r.normal(n, case["k"], std=0.02, dtype=dt) for n in _parts(case)]
    bs = [r.normal(n, std=0.01, dtype=dt) if case["bias"] else None for n in _parts(case)]
    return x, ws, bs


def _conv_inputs(case, seed):
    r = _Rand(seed)
    dt = case["dtype"]
    x = r.normal(case["n"], case["ci"], case["h"], case["w"], dtype=dt)
    w = r.normal(case["co"], case["ci"], 3, 3, std=0.02, dtype=dt)
    return x, w, r.normal(case["co"], std=0.01, dtype=dt) if case["bias"] else None


def _chain_inputs(case, seed):
    r = _Rand(seed)
    dt = case["dtype"]
    x = r.normal(case["n"], case["ci"], case["h"], case["w"], dtype=dt)
    ws, bs, ci = [], [], case["ci"]
    for co, _ in _chain(case):
        ws.append(r.conv(co, ci, dt))
        bs.append(r.normal(co, std=0.01, dtype=dt) if case["bias"] else None)
        ci = co
    return x, ws, bs


def _attention_inputs(case, seed):
    r = _Rand(seed)
    T = sum(_lens(case))
    return (r.normal(T, NH, DH, dtype="bf16"), r.normal(T, NKV, DH, dtype="bf16"), r.normal(T, NKV, DH, dtype="bf16"))


def _stack_inputs(case, seed):
    r = _Rand(seed)
    lens = _lens(case)
    weights = {}
    for i in range(case["layers"]):
        for key in stack.LAYER_KEYS:
            shape = stack.LAYER_SHAPES[key]
            if len(shape) == 2:
                weights[(i, key)] = r.normal(*shape, std=0.02, dtype="bf16")
            else:
                weights[(i, key)] = (1 + 0.1 * r.normal(*shape)).to(torch.bfloat16)
    weights["norm"] = (1 + 0.1 * r.normal(D)).to(torch.bfloat16)
    weights["head"] = r.normal(case["out"], D, std=0.02, dtype="bf16")
    weights["inv_freq"] = (1.0 / 1e6 ** (torch.arange(0, DH, 2, dtype=torch.float32) / DH)).to(r.dev)
    L = max(lens)
    mask = torch.zeros(len(lens), 1, L, L, dtype=torch.bool, device=r.dev)
    for b, n in enumerate(lens):
        mask[b, :, :n, :n] = True
        i = torch.arange(n, L, device=r.dev)
        mask[b, :, i, i] = True
    return r.normal(len(lens), L, D), mask, weights


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, ws, bs = _linear_inputs(case, seed)
        return {"kind": kind, "x": x, "ws": ws, "bs": bs, "cid": _config(case["precision"])}
    if kind == "conv":
        x, w, b = _conv_inputs(case, seed)
        return {"kind": kind, "x": x, "w": w, "b": b, "relu": case["relu"], "cid": _config()}
    if kind == "chain":
        x, ws, bs = _chain_inputs(case, seed)
        layers = _chain(case)
        # without biases the ReLU is the conv's own (unsigned saturation), with them it follows the bias
        return {"kind": kind, "x": x, "ws": ws, "bs": bs, "relus": [not case["bias"]] * len(layers),
                "after": [case["bias"]] * len(layers), "pools": [p for _, p in layers], "cid": _config()}
    if kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        lens = _lens(case)
        cols = [kernels.round_up(n, 32) for n in lens]
        starts = [sum(lens[:b]) for b in range(len(lens))]
        vts = [sum(cols[:b]) for b in range(len(lens))]
        vt = torch.zeros(NKV, DH, sum(cols), dtype=torch.bfloat16, device=q.device)
        for n, s, c in zip(lens, starts, vts):
            vt[:, :, c:c + n] = v[s:s + n].permute(1, 2, 0)
        meta = [torch.tensor(m, dtype=torch.int32, device=q.device) for m in (starts, lens, vts)]
        return {"kind": kind, "q": q, "k": k, "vt": vt, "meta": meta, "longest": max(lens)}
    x, mask, weights = _stack_inputs(case, seed)
    sid = stack.register(stack.Plan([], None, None, 1, None, weights, None, case["layers"], case["out"],
                                    stack.MAX_TOKENS))
    return {"kind": kind, "x": x, "mask": mask, "weights": weights, "sid": sid, "cid": _config()}


def run(state):
    s, kind = state, state["kind"]
    with torch.no_grad():
        if kind == "linear":
            if len(s["ws"]) == 1:
                return torch.ops.xdna.linear(s["x"], s["ws"][0], s["bs"][0], False, s["cid"])
            return torch.ops.xdna.linear_cat(s["x"], s["ws"], s["bs"], s["cid"])
        if kind == "conv":
            return torch.ops.xdna.conv3x3_fused(s["x"], s["w"], s["b"], s["relu"], s["cid"])
        if kind == "chain":
            return torch.ops.xdna.conv3x3_chain(s["x"], s["ws"], s["bs"], s["relus"], s["after"], s["pools"], s["cid"])
        if kind == "attention":
            return kernels.attention_bf16(s["q"], s["k"], s["vt"], *s["meta"], s["longest"], DH ** -0.5)
        return torch.ops.xdna.qwen3_stack(s["x"], s["mask"], s["sid"], s["cid"])


# ------------------------------------------------------------------------------ what a pass cannot do without
def _stack_params(case):
    return case["layers"] * (D * (NH + 2 * NKV) * DH + NH * DH * D + 3 * D * INTER) + D * case["out"]


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n, esz = case["m"], case["k"], sum(_parts(case)), ESZ[case["dtype"]]
        wsz = 2 if case["precision"] == "bf16" else 1
        return {"bytes": (m * k + m * n) * esz + n * k * wsz + 4 * n + (esz * n if case["bias"] else 0),
                "flops": 2 * m * n * k}
    if kind == "conv":
        px, esz = case["n"] * case["h"] * case["w"], ESZ[case["dtype"]]
        return {"bytes": px * (case["ci"] + case["co"]) * esz + 9 * case["ci"] * case["co"],
                "flops": 18 * px * case["ci"] * case["co"]}
    if kind == "chain":
        h, w, ci, esz = case["h"], case["w"], case["ci"], ESZ[case["dtype"]]
        total, flops = case["n"] * h * w * ci * esz, 0
        for i, (co, pool) in enumerate(_chain(case)):
            total += 9 * ci * co
            flops += 18 * case["n"] * h * w * ci * co
            out, ci = case["n"] * h * w * co * esz, co
            if pool:
                h, w = h // 2, w // 2
        return {"bytes": total + out, "flops": flops}
    lens = _lens(case)
    attn = sum(4 * n * n * NH * DH for n in lens)
    if kind == "attention":
        return {"bytes": sum(lens) * (2 * NH + 2 * NKV) * DH * 2, "flops": attn}
    T = len(lens) * max(lens)
    return {"bytes": 2 * _stack_params(case) + 4 * T * (D + case["out"]),
            "flops": 2 * sum(lens) * _stack_params(case) + case["layers"] * attn}


def tolerance(case):
    """The int8 ops promise the reference's integers and its float32 steps after them, bit for bit. The
    others multiply bf16 values in the order a kernel likes: measured against `exact` and stated about
    four times as wide."""
    kind = case["kind"]
    if kind == "attention":
        return {"rel": 1e-2, "max": 0.05}     # probabilities and outputs rounded to bf16
    if kind == "stack":
        return {"rel": 2e-2, "max": 0.1}      # bf16 operands through every layer
    if kind == "linear" and case["precision"] == "bf16":
        # float32 sums of bf16 products, rounded once to the output's dtype
        return {"rel": {"f32": 4e-6, "f16": 5e-4, "bf16": 4e-3}[case["dtype"]],
                "max": {"f32": 1e-4, "f16": 2e-3, "bf16": 2e-2}[case["dtype"]]}
    return "exact"


# ------------------------------------------------------------------------------ in 64 bits
def _quantized(x, dims):
    """(integers, scale) of symmetric int8: scale = max |x| / 127 and x / scale in float32, as the op is
    defined (the quotients of two float32 numbers, rounded once through float64); integers as float64."""
    amax = x.float().abs().amax(dim=dims, keepdim=True).clamp(min=1e-8)
    s = (amax.double() / 127).float()
    return torch.round((x.double() / s.double()).float()).clamp(-127, 127).double(), s


def _conv_sums(q, wq):
    """3x3, padding 1, of whole numbers in float64 (exact), as nine products."""
    n, ci, h, w = q.shape
    p = F.pad(q, (1, 1, 1, 1))
    out = torch.zeros(n, wq.shape[0], h * w, dtype=torch.float64, device=q.device)
    for ky in range(3):
        for kx in range(3):
            win = p[:, :, ky:ky + h, kx:kx + w].reshape(n, ci, h * w)
            tap = wq[:, :, ky, kx].contiguous()
            for b in range(n):
                out[b].addmm_(tap, win[b])
    return out.view(n, -1, h, w)


def _conv_layer(x, weight, relu):
    """(requantized integers, scale [1, co, 1, 1], sx [n, 1, 1, 1]) of one conv's first call."""
    q, sx = _quantized(x, (1, 2, 3))
    wq, sw = _quantized(weight, (1, 2, 3))
    acc = _conv_sums(q, wq)
    top = float(acc[0].clamp(min=0).max() if relu else acc[0].abs().max())
    shift = min(31, max(1, math.ceil(math.log2(max(top * 1.25, 1.0) / (255 if relu else 127)))))
    r = torch.floor((acc + 2.0 ** (shift - 1)) / 2.0 ** shift)
    return r.clamp(0, 255) if relu else r.clamp(-128, 127), sw.view(1, -1, 1, 1) * 2.0 ** shift, sx


def _dequantized(r, scale, sx, bias, wide):
    """r * (scale * sx) (+ bias): in float64 (`wide`, the last layer) or as the float32 steps the next layer
    sees."""
    y = r * (scale.double() * sx.double()) if wide else (r * (scale * sx).double()).float()
    if bias is not None:
        y = y + bias.to(y.dtype).view(1, -1, 1, 1)
    return y


def _rms(x, w, eps=1e-6):
    return w.double() * (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps))


def _attend(q, k, v):
    """q [n, NH, DH], k and v [n, NKV, DH] in float64, one sequence."""
    q = q.permute(1, 0, 2).reshape(NKV, NH // NKV, -1, DH)
    k, v = k.permute(1, 2, 0), v.permute(1, 0, 2)
    out = []
    for g in range(NKV):
        for h in range(NH // NKV):
            out.append(torch.softmax((q[g, h] @ k[g]) * DH ** -0.5, dim=-1) @ v[g])
    return torch.stack(out, 1)


def _rope(x, ang):
    c, s = ang.cos().double()[:, None], ang.sin().double()[:, None]
    a, b = x[..., :DH // 2], x[..., DH // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _stack_exact(case, seed):
    x, _, W = _stack_inputs(case, seed)
    lens = _lens(case)
    B, L = x.shape[:2]
    X = torch.cat([x[b, :n] for b, n in enumerate(lens)]).double()
    pos = torch.cat([torch.arange(n, device=x.device) for n in lens])
    ang = pos.float()[:, None] * W["inv_freq"][None]
    T = X.shape[0]
    for i in range(case["layers"]):
        w = {key: W[(i, key)].double() for key in stack.LAYER_KEYS}
        h = _rms(X, w["input_norm"])
        q = _rope(_rms((h @ w["q"].t()).view(T, NH, DH), w["q_norm"]), ang)
        k = _rope(_rms((h @ w["k"].t()).view(T, NKV, DH), w["k_norm"]), ang)
        v = (h @ w["v"].t()).view(T, NKV, DH)
        at, s = [], 0
        for n in lens:
            at.append(_attend(q[s:s + n], k[s:s + n], v[s:s + n]).reshape(n, NH * DH))
            s += n
        X = X + torch.cat(at) @ w["o"].t()
        h = _rms(X, w["post_norm"])
        X = X + (F.silu(h @ w["gate"].t()) * (h @ w["up"].t())) @ w["down"].t()
    y = _rms(X, W["norm"]) @ W["head"].double().t()
    out = torch.zeros(B, L, case["out"], dtype=torch.float64, device=x.device)
    s = 0
    for b, n in enumerate(lens):
        out[b, :n] = y[s:s + n]
        s += n
    return out


def exact(case, seed):
    """What `run` returns in 64 bits. The int8 of an activation is part of what the ops are (the float32
    scale and quotient), and so are a chain's float values between its layers; everything else (sums,
    products of the scales' values, biases, softmax, norms) is float64."""
    with torch.no_grad():
        kind = case["kind"]
        if kind == "linear":
            x, ws, bs = _linear_inputs(case, seed)
            if case["precision"] == "bf16":
                y = x.bfloat16().double() @ torch.cat(ws).bfloat16().double().t()
            else:
                q, sx = _quantized(x, (1,))
                wq, sw = _quantized(torch.cat(ws), (1,))
                y = (q @ wq.t()) * sx.double() * sw.double().view(1, -1)
            return y + torch.cat(bs).double() if case["bias"] else y
        if kind == "conv":
            x, w, b = _conv_inputs(case, seed)
            return _dequantized(*_conv_layer(x, w, case["relu"]), b, True)
        if kind == "chain":
            x, ws, bs = _chain_inputs(case, seed)
            layers = _chain(case)
            for i, (_, pool) in enumerate(layers):
                last = i == len(layers) - 1
                y = _dequantized(*_conv_layer(x, ws[i], not case["bias"]), bs[i], last)
                if not last:
                    x = torch.relu(y.to(DTYPES[case["dtype"]]))
                    x = F.max_pool2d(x, 2, 2) if pool else x
            return y
        if kind == "attention":
            q, k, v = (t.double() for t in _attention_inputs(case, seed))
            out, s = [], 0
            for n in _lens(case):
                out.append(_attend(q[s:s + n], k[s:s + n], v[s:s + n]))
                s += n
            return torch.cat(out)
        return _stack_exact(case, seed)
