"""The work that a user of this framework has it do, as measurable cases.

Every case is one pass through the public functions of teenygrad_amd.kernels
on device buffers that the program keeps, on the null stream, with the one
operator workspace that the program attached to it when it started.

The cases stand for (`op`):

  conv_f32       fp32 NCHW conv + bias + ReLU at small batch: the reference's
                 own conv call, a few microseconds of work where launches and
                 latency count
  norm_act       LayerNorm -> GELU and RMSNorm -> SiLU of one tensor, bf16 or
                 fp32: the bandwidth-bound chain of a transformer block
  mlp_train      forward and backward of a transformer's MLP block in bf16:
                 LayerNorm, linear, GELU, linear and all their gradients
  attn_prefill   bf16 attention over whole prompts (causal), or of a prompt
                 against a longer context, with or without grouped K/V heads
  attn_decode    bf16 attention of one or a few new queries per sequence
                 against its cached K/V: generation, one token at a time
  attn_train     bf16 attention forward and backward
  attn_f32       fp32 attention forward and backward: the reference's type
  resnet_block   a ResNet-50 bottleneck (1x1, 3x3, 1x1, BatchNorm folded into
                 the biases) in bf16 NHWC, or with int8 weights
  conv_train     forward, dx and dw of one ResNet-50 conv in bf16 NHWC
  w8a16_prefill  a quantized MLP (int8 weights, bf16 activations) over the
                 tokens of whole prompts: compute-bound
  w8a16_decode   the same MLP for one token of each of a few sequences: bound
                 by reading the weights
  linear_f32     forward and backward of an fp32 linear layer with bias

Inputs are made from the seed alone, by a generator on the device.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

import teenygrad_amd as tg
from teenygrad_amd import kernels as K
from teenygrad_amd.runtime import NULL_STREAM

WORKSPACE = 256 << 20  # one scratch buffer for every operator of the program's stream


def listed():
    return [
        # one image through the conv + ReLU that the reference's tests and book time
        {"name": "conv_f32_56x56", "op": "conv_f32", "b": 1, "cin": 64, "cout": 64, "h": 56, "w": 56, "k": 3, "s": 1},
        # norms and activations of 16384 tokens of width 4096
        {"name": "norm_act_bf16", "op": "norm_act", "m": 16384, "n": 4096, "dtype": "bf16"},
        # a training step of a 1024-wide MLP block on 2000 tokens (a ragged batch)
        {"name": "mlp_train_1024", "op": "mlp_train", "m": 2000, "h": 1024, "f": 4096},
        # eight prompts of 2048 tokens, 32 heads
        {"name": "attn_prefill_2048", "op": "attn_prefill", "b": 8, "hq": 32, "hkv": 32, "nq": 2048, "nk": 2048,
         "d": 128, "causal": True},
        # sixteen sequences, each with 4000 tokens of context, grouped K/V heads
        {"name": "attn_decode_4000", "op": "attn_decode", "b": 16, "hq": 32, "hkv": 8, "nq": 1, "nk": 4000, "d": 128,
         "causal": False},
        # training at an ordinary context length, head size 64
        {"name": "attn_train_1024", "op": "attn_train", "b": 4, "hq": 16, "hkv": 16, "nq": 1024, "nk": 1024, "d": 64,
         "causal": True},
        # fp32 at a ragged length
        {"name": "attn_f32_500", "op": "attn_f32", "b": 2, "hq": 8, "hkv": 8, "nq": 500, "nk": 500, "d": 64,
         "causal": False},
        # stage 3 of ResNet-50 at batch 16
        {"name": "resnet_block_14x14", "op": "resnet_block", "b": 16, "width": 256, "cin": 1024, "h": 14, "s": 1,
         "weights": "bf16"},
        # stage 2's 3x3 conv in training at batch 32
        {"name": "conv_train_28x28", "op": "conv_train", "b": 32, "cin": 128, "cout": 128, "h": 28, "k": 3, "s": 1},
        # 4096 prompt tokens through a 4096-wide MLP
        {"name": "w8a16_prefill_4096", "op": "w8a16_prefill", "m": 4096, "h": 4096, "f": 11008},
        # one token of each of eight sequences through the same MLP
        {"name": "w8a16_decode_8", "op": "w8a16_decode", "m": 8, "h": 4096, "f": 11008},
        # an fp32 layer of ordinary width
        {"name": "linear_f32_1024", "op": "linear_f32", "m": 1000, "n": 1024, "k": 1024},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _of8(rng, low, high):
    return max(low, 8 * round(_log(rng, low, high) / 8))


def _draw_attention(rng, op):
    d = rng.choice([64, 128])
    hkv = rng.choice([1, 2, 4, 8, 16, 32])
    hq = hkv * rng.choice([1, 1, 2, 4, 8])
    if op == "attn_decode":
        return {"op": op, "b": _log(rng, 1, 64), "hq": hq, "hkv": hkv, "nq": rng.choice([1, 1, 1, 2, 5]),
                "nk": _log(rng, 64, 16384), "d": d, "causal": False}
    if op == "attn_f32":
        d, hq = rng.choice([16, 32, 64, 128]), hkv
    nq = _log(rng, 16, 1024) if op == "attn_f32" else _log(rng, 64, 4096)
    causal = rng.random() < 0.6
    nk = nq if causal or rng.random() < 0.5 else _log(rng, 16, 1024 if op == "attn_f32" else 4096)
    return {"op": op, "b": _log(rng, 1, 16), "hq": hq, "hkv": hkv, "nq": nq, "nk": nk, "d": d, "causal": causal}


def _draw(rng, op):
    if op == "conv_f32":
        k = rng.choice([1, 3, 3, 5])
        return {"op": op, "b": _log(rng, 1, 8), "cin": rng.choice([3, 16, 32, 64, 100, 128, 256]),
                "cout": rng.choice([16, 32, 48, 64, 128, 256]), "h": _log(rng, 7, 112), "w": _log(rng, 7, 112), "k": k,
                "s": rng.choice([1, 1, 2])}
    if op == "norm_act":
        n = _log(rng, 64, 8192)
        return {"op": op, "m": _log(rng, 1, 16384), "n": n if rng.random() < 0.3 else max(64, 64 * round(n / 64)),
                "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if op == "mlp_train":
        h = max(128, 64 * round(_log(rng, 128, 2048) / 64))
        return {"op": op, "m": _log(rng, 32, 8192), "h": h, "f": rng.choice([2, 3, 4]) * h}
    if op.startswith("attn"):
        return _draw_attention(rng, op)
    if op in ("resnet_block", "conv_train"):
        stage = rng.randrange(4)
        width, h = 64 << stage, 56 >> stage
        s = rng.choice([1, 1, 2]) if stage else 1
        b = _log(rng, 1, 64)
        if op == "resnet_block":  # a stage's first block strides and reads the stage before
            return {"op": op, "b": b, "width": width, "cin": 2 * width if s == 2 else 4 * width, "h": h * s, "s": s,
                    "weights": rng.choice(["bf16", "bf16", "int8"])}
        k = rng.choice([1, 3])
        cin, cout = (width, width) if k == 3 else rng.choice([(width, 4 * width), (4 * width, width)])
        return {"op": op, "b": b, "cin": cin, "cout": cout, "h": h * s, "k": k, "s": s}
    if op in ("w8a16_prefill", "w8a16_decode"):
        h = max(512, 128 * round(_log(rng, 512, 8192) / 128))
        f = max(512, 64 * round(h * rng.choice([2.6875, 3.5, 4]) / 64))
        return {"op": op, "m": _log(rng, 1, 64) if op == "w8a16_decode" else _log(rng, 128, 8192), "h": h, "f": f}
    return {"op": op, "m": _log(rng, 1, 4096), "n": _log(rng, 10, 4096), "k": _log(rng, 16, 4096)}


def draw(rng):
    op = rng.choice([c["op"] for c in listed()])
    most = {c["op"]: work(c) for c in listed()}
    top = max(w["bytes"] for w in most.values())
    while True:  # no dearer than the listed case of its kind, but for twice its bytes
        case = _draw(rng, op)
        cost = work(case)
        if cost["flops"] <= most[op]["flops"] and cost["bytes"] <= min(top, 2 * most[op]["bytes"]):
            return case


# ── what the program holds ──────────────────────────────────────────────────

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "i8": torch.int8}
_TYPESTR = {"f32": "<f4", "bf16": "<i2", "i8": "|i1"}


class _Array:
    """A framework buffer as torch sees it (no copy; keeps the buffer alive)."""

    def __init__(self, buf):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": buf.shape, "typestr": _TYPESTR[buf.dtype.name],
                                         "data": (buf.ptr, False), "version": 3}


def _view(buf):
    t = torch.as_tensor(_Array(buf), device="cuda")
    return t.view(torch.bfloat16) if buf.dtype.name == "bf16" else t


def _conv(case):
    """(padding, output height, output width) of a conv case."""
    p = case["k"] // 2
    h, w = case["h"], case.get("w", case["h"])
    return p, (h + 2 * p - case["k"]) // case["s"] + 1, (w + 2 * p - case["k"]) // case["s"] + 1


def _shapes(case):
    """({input: (dtype, shape, mean, deviation)}, {output: (dtype, shape)}) of a case."""
    op = case["op"]
    if op == "conv_f32":
        b, ci, co, k = case["b"], case["cin"], case["cout"], case["k"]
        _, oh, ow = _conv(case)
        return ({"x": ("f32", (b, ci, case["h"], case["w"]), 0, 1),
                 "w": ("f32", (co, ci, k, k), 0, math.sqrt(2 / (ci * k * k))), "bias": ("f32", (co,), 0, 0.01)},
                {"y": ("f32", (b, co, oh, ow))})
    if op == "norm_act":
        t, x = case["dtype"], (case["m"], case["n"])
        n = (case["n"],)
        return ({"x": (t, x, 0, 1), "gamma": (t, n, 1, 0.02), "beta": (t, n, 0, 0.02), "weight": (t, n, 1, 0.02)},
                {k: (t, x) for k in ("ln", "gelu", "rms", "silu")})
    if op == "mlp_train":
        m, h, f = case["m"], case["h"], case["f"]
        return ({"x": ("bf16", (m, h), 0, 1), "gamma": ("bf16", (h,), 1, 0.02), "beta": ("bf16", (h,), 0, 0.02),
                 "w1": ("bf16", (f, h), 0, 1 / math.sqrt(h)), "b1": ("bf16", (f,), 0, 0.02),
                 "w2": ("bf16", (h, f), 0, 1 / math.sqrt(f)), "b2": ("bf16", (h,), 0, 0.02),
                 "do": ("bf16", (m, h), 0, 1)},
                {"y": ("bf16", (m, h)), "mean": ("f32", (m,)), "rstd": ("f32", (m,)), "h": ("bf16", (m, f)),
                 "a": ("bf16", (m, f)), "o": ("bf16", (m, h)), "da": ("bf16", (m, f)), "dw2": ("bf16", (h, f)),
                 "db2": ("bf16", (h,)), "dh": ("bf16", (m, f)), "dy": ("bf16", (m, h)), "dw1": ("bf16", (f, h)),
                 "db1": ("bf16", (f,)), "dx": ("bf16", (m, h)), "dgamma": ("f32", (h,)), "dbeta": ("f32", (h,))})
    if op.startswith("attn"):
        t = "f32" if op == "attn_f32" else "bf16"
        q = (case["b"] * case["hq"], case["nq"], case["d"])
        kv = (case["b"] * case["hkv"], case["nk"], case["d"])
        ins = {"q": (t, q, 0, 1), "k": (t, kv, 0, 1), "v": (t, kv, 0, 1)}
        outs = {"o": (t, q)}
        if op in ("attn_train", "attn_f32"):
            ins["do"] = (t, q, 0, 1)
            outs.update(lse=("f32", q[:2]), dq=(t, q), dk=(t, kv), dv=(t, kv))
        return ins, outs
    if op == "resnet_block":
        b, c, ci, h, s = case["b"], case["width"], case["cin"], case["h"], case["s"]
        oh = (h - 1) // s + 1
        i8 = case["weights"] == "int8"
        ins = {"x": ("bf16", (b, h, h, ci), 0, 1)}
        for n, co, k, fan in (("1", c, 1, ci), ("2", c, 3, c), ("3", 4 * c, 1, c)):
            ins["w" + n] = ("i8" if i8 else "bf16", (co, k, k, fan), 0, math.sqrt(2 / (fan * k * k)))
            ins["b" + n] = ("f32" if i8 else "bf16", (co,), 0, 0.1)
        return ins, {"c1": ("bf16", (b, h, h, c)), "c2": ("bf16", (b, oh, oh, c)), "c3": ("bf16", (b, oh, oh, 4 * c))}
    if op == "conv_train":
        b, ci, co, h, k = case["b"], case["cin"], case["cout"], case["h"], case["k"]
        _, oh, ow = _conv(case)
        x, w, y = (b, h, h, ci), (co, k, k, ci), (b, oh, ow, co)
        return ({"x": ("bf16", x, 0, 1), "w": ("bf16", w, 0, math.sqrt(2 / (ci * k * k))), "dy": ("bf16", y, 0, 1)},
                {"y": ("bf16", y), "dx": ("bf16", x), "dw": ("bf16", w)})
    if op in ("w8a16_prefill", "w8a16_decode"):
        m, h, f = case["m"], case["h"], case["f"]
        return ({"x": ("bf16", (m, h), 0, 1), "up": ("i8", (f, h), 0, 0.02), "down": ("i8", (h, f), 0, 0.02)},
                {"h": ("bf16", (m, f)), "y": ("bf16", (m, h))})
    m, n, k = case["m"], case["n"], case["k"]
    return ({"x": ("f32", (m, k), 0, 1), "w": ("f32", (n, k), 0, 1 / math.sqrt(k)), "b": ("f32", (n,), 0, 0.02),
             "dy": ("f32", (m, n), 0, 1)},
            {"y": ("f32", (m, n)), "dx": ("f32", (m, k)), "dw": ("f32", (n, k)), "db": ("f32", (n,))})


def _inputs(case, seed):
    """The input tensors; an int8 weight comes with its fp32 scales (per output channel, symmetric)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    made = {}
    for name, (dtype, shape, mean, std) in _shapes(case)[0].items():
        t = torch.randn(shape, generator=gen, device="cuda").mul_(std).add_(mean)
        if dtype == "i8":
            flat = t.flatten(1)
            scale = flat.abs().amax(1) / 127
            made[name + "_scale"] = scale
            t = (flat / scale[:, None]).round_().reshape(shape)
        made[name] = t.to(_TORCH[dtype])
    return made


_NAMES = {v: k for k, v in _TORCH.items()}


def prepare(case, seed):
    dev = tg.open(0)
    if NULL_STREAM._workspace is None:
        NULL_STREAM.set_workspace(dev.buffer(tg.i8, (WORKSPACE,)))
    bufs = {}
    for name, t in _inputs(case, seed).items():
        bufs[name] = dev.buffer(_NAMES[t.dtype], tuple(t.shape))
        _view(bufs[name]).copy_(t)
    outs = {n: dev.buffer(d, s) for n, (d, s) in _shapes(case)[1].items()}
    return {"case": case, "in": bufs, "out": outs, "views": {n: _view(o) for n, o in outs.items()}}


# ── one pass ────────────────────────────────────────────────────────────────


def _run_conv_f32(c, i, o):
    K.conv2d(i["x"], i["w"], i["bias"], stride=c["s"], padding=c["k"] // 2, act="relu", y=o["y"])


def _run_norm_act(c, i, o):
    K.layer_norm(i["x"], i["gamma"], i["beta"], 1e-5, y=o["ln"])
    K.gelu(o["ln"], o["gelu"])
    K.rms_norm(i["x"], i["weight"], 1e-8, y=o["rms"])
    K.silu(o["rms"], o["silu"])


def _run_mlp_train(c, i, o):
    K.layer_norm_train(i["x"], i["gamma"], i["beta"], 1e-5, y=o["y"], mean=o["mean"], rstd=o["rstd"])
    K.linear(o["y"], i["w1"], i["b1"], y=o["h"])
    K.gelu(o["h"], o["a"])
    K.linear(o["a"], i["w2"], i["b2"], y=o["o"])
    K.linear_backward(o["a"], i["w2"], i["do"], dx=o["da"], dw=o["dw2"], db=o["db2"])
    K.gelu_backward(o["da"], o["h"], o["dh"])
    K.linear_backward(o["y"], i["w1"], o["dh"], dx=o["dy"], dw=o["dw1"], db=o["db1"])
    o["dgamma"].zero_()
    o["dbeta"].zero_()
    K.layer_norm_backward(o["dy"], i["x"], i["gamma"], o["mean"], o["rstd"], o["dgamma"], o["dbeta"], dx=o["dx"])


def _run_attention(c, i, o):
    K.attention(i["q"], i["k"], i["v"], c["hq"], c["hkv"], causal=c["causal"], o=o["o"], lse=o.get("lse"))
    if "dq" in o:
        K.attention_backward(i["q"], i["k"], i["v"], o["o"], i["do"], o["lse"], c["hq"], c["hkv"], causal=c["causal"],
                             dq=o["dq"], dk=o["dk"], dv=o["dv"])


def _run_resnet_block(c, i, o):
    def conv(n, x, y, s, p, act):
        if c["weights"] == "int8":
            K.w8a16_conv2d(x, i["w" + n], i["w" + n + "_scale"], i["b" + n], stride=s, padding=p, act=act, y=y)
        else:
            K.conv2d(x, i["w" + n], i["b" + n], stride=s, padding=p, act=act, layout="nhwc", y=y)

    conv("1", i["x"], o["c1"], 1, 0, "relu")
    conv("2", o["c1"], o["c2"], c["s"], 1, "relu")
    conv("3", o["c2"], o["c3"], 1, 0, None)


def _run_conv_train(c, i, o):
    opt = {"stride": c["s"], "padding": c["k"] // 2, "layout": "nhwc"}
    K.conv2d(i["x"], i["w"], y=o["y"], **opt)
    K.conv2d_backward_dx(i["dy"], i["w"], i["x"].shape, dx=o["dx"], **opt)
    K.conv2d_backward_dw(i["dy"], i["x"], i["w"].shape, dw=o["dw"], **opt)


def _run_w8a16(c, i, o):
    K.w8a16_linear(i["x"], i["up"], i["up_scale"], act="silu", y=o["h"])
    K.w8a16_linear(o["h"], i["down"], i["down_scale"], y=o["y"])


def _run_linear_f32(c, i, o):
    K.linear(i["x"], i["w"], i["b"], y=o["y"])
    K.linear_backward(i["x"], i["w"], i["dy"], dx=o["dx"], dw=o["dw"], db=o["db"])


_RUN = {"conv_f32": _run_conv_f32, "norm_act": _run_norm_act, "mlp_train": _run_mlp_train,
        "attn_prefill": _run_attention, "attn_decode": _run_attention, "attn_train": _run_attention,
        "attn_f32": _run_attention, "resnet_block": _run_resnet_block, "conv_train": _run_conv_train,
        "w8a16_prefill": _run_w8a16, "w8a16_decode": _run_w8a16, "linear_f32": _run_linear_f32}


def run(state):
    _RUN[state["case"]["op"]](state["case"], state["in"], state["out"])
    return state["views"]


# ── what a pass cannot do without ───────────────────────────────────────────

_SIZE = {"f32": 4, "bf16": 2, "i8": 1}


def work(case):
    ins, outs = _shapes(case)
    size = sum(_SIZE[t[0]] * int(np.prod(t[1])) for t in (*ins.values(), *outs.values()))
    op = case["op"]
    if op == "conv_f32":
        _, oh, ow = _conv(case)
        flops = 2 * case["b"] * case["cout"] * oh * ow * case["cin"] * case["k"] ** 2
    elif op == "norm_act":
        flops = 30 * case["m"] * case["n"]
    elif op == "mlp_train":
        flops = 12 * case["m"] * case["h"] * case["f"]
    elif op.startswith("attn"):
        pairs = case["nq"] * case["nk"]
        if case["causal"]:  # query i meets the keys up to i
            n = min(case["nq"], case["nk"])
            pairs = n * (n + 1) // 2 + (case["nq"] - n) * case["nk"]
        flops = 4 * case["b"] * case["hq"] * pairs * case["d"] * (3.5 if "do" in ins else 1)
    elif op == "resnet_block":
        c, h, oh = case["width"], case["h"], (case["h"] - 1) // case["s"] + 1
        flops = 2 * case["b"] * (h * h * case["cin"] * c + oh * oh * (9 * c * c + 4 * c * c))
    elif op == "conv_train":
        _, oh, ow = _conv(case)
        flops = 6 * case["b"] * oh * ow * case["cin"] * case["cout"] * case["k"] ** 2
    elif op.startswith("w8a16"):
        flops = 4 * case["m"] * case["h"] * case["f"]
    else:
        flops = 6 * case["m"] * case["n"] * case["k"]
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """About four times the error against `exact` (2-norm, worst output) that the path shows: at most 1e-6 in fp32,
    2.6e-3 behind one or two bf16 roundings, 2.9e-3 at the end of a ResNet block and 3.6e-3 at that of the MLP step."""
    op = case["op"]
    if op in ("conv_f32", "attn_f32", "linear_f32") or case.get("dtype") == "f32":
        return {"rel": 4e-6}
    return {"rel": {"mlp_train": 1.5e-2, "resnet_block": 1.2e-2}.get(op, 1e-2)}


# ── the same in 64 bits ─────────────────────────────────────────────────────


def _attention64(case, t):
    """o (and lse and the gradients) over a few K/V heads at a time."""
    group = case["hq"] // case["hkv"]
    bkv, nq, nk, d = case["b"] * case["hkv"], case["nq"], case["nk"], case["d"]
    train = "do" in t
    q = t["q"].reshape(bkv, group * nq, d)
    do = t["do"].reshape(bkv, group * nq, d) if train else None
    mask = torch.ones(nq, nk, dtype=torch.bool, device=q.device).tril().repeat(group, 1) if case["causal"] else None
    made = {n: [] for n in (("o", "lse", "dq", "dk", "dv") if train else ("o",))}
    step = max(1, (1 << 27) // (group * nq * nk))
    for a in range(0, bkv, step):
        qa, ka, va = (x[a:a + step].double() for x in (q, t["k"], t["v"]))
        s = torch.bmm(qa, ka.mT.contiguous()) / math.sqrt(d)
        if mask is not None:
            s.masked_fill_(~mask, -math.inf)
        lse = torch.logsumexp(s, -1)
        p = torch.exp(s - lse[..., None])
        o = torch.bmm(p, va)
        made["o"].append(o)
        if train:
            g = do[a:a + step].double()
            ds = torch.bmm(g, va.mT.contiguous()).sub_((g * o).sum(-1, keepdim=True)).mul_(p).div_(math.sqrt(d))
            made["lse"].append(lse)
            made["dq"].append(torch.bmm(ds, ka))
            made["dk"].append(torch.bmm(ds.mT.contiguous(), qa))
            made["dv"].append(torch.bmm(p.mT.contiguous(), g))
    made = {n: torch.cat(v) for n, v in made.items()}
    for n in ("o", "dq"):
        if n in made:
            made[n] = made[n].reshape(t["q"].shape)
    if train:
        made["lse"] = made["lse"].reshape(t["q"].shape[:2])
    return made


def _conv64(x, w, bias, s, p):
    """NHWC conv as one product per tap."""
    co, kh, kw, ci = w.shape
    b, h, wd, _ = x.shape
    oh, ow = (h + 2 * p - kh) // s + 1, (wd + 2 * p - kw) // s + 1
    x = F.pad(x, (0, 0, p, p, p, p))
    y = torch.zeros(b * oh * ow, co, dtype=torch.float64, device=x.device)
    for a in range(kh):
        for c in range(kw):
            tap = x[:, a:a + s * (oh - 1) + 1:s, c:c + s * (ow - 1) + 1:s].reshape(-1, ci)
            y = y + tap @ w[:, a, c].T.contiguous()
    y = y.reshape(b, oh, ow, co)
    return y if bias is None else y + bias


def _linear_grads64(x, w, dy):
    return dy @ w, dy.T.contiguous() @ x, dy.sum(0)


def exact(case, seed):
    op = case["op"]
    t = _inputs(case, seed)
    if op.startswith("attn"):
        return _attention64(case, t)
    t = {n: v.double() for n, v in t.items()}
    if op == "conv_f32":
        y = _conv64(t["x"].permute(0, 2, 3, 1), t["w"].permute(0, 2, 3, 1), t["bias"], case["s"], case["k"] // 2)
        return {"y": y.relu().permute(0, 3, 1, 2).contiguous()}
    if op == "norm_act":
        x, n = t["x"], (case["n"],)
        ln = F.layer_norm(x, n, t["gamma"], t["beta"], 1e-5)
        rms = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-8) * t["weight"]
        return {"ln": ln, "gelu": F.gelu(ln, approximate="tanh"), "rms": rms, "silu": F.silu(rms)}
    if op == "mlp_train":
        x, g = t["x"], t["gamma"]
        mean = x.mean(-1)
        rstd = torch.rsqrt(x.var(-1, unbiased=False) + 1e-5)
        xhat = (x - mean[:, None]) * rstd[:, None]
        y = xhat * g + t["beta"]
        h = y @ t["w1"].T.contiguous() + t["b1"]
        h.requires_grad_()
        a = F.gelu(h, approximate="tanh")
        da, dw2, db2 = _linear_grads64(a.detach(), t["w2"], t["do"])
        dh, = torch.autograd.grad(a, h, da)
        h, a = h.detach(), a.detach()
        dy, dw1, db1 = _linear_grads64(y, t["w1"], dh)
        # the reference's form: gamma outside the bracket as well
        c1, c2 = (dy * g).mean(-1, keepdim=True), (dy * g * xhat).mean(-1, keepdim=True)
        return {"y": y, "mean": mean, "rstd": rstd, "h": h, "a": a, "o": a @ t["w2"].T.contiguous() + t["b2"],
                "da": da, "dw2": dw2, "db2": db2, "dh": dh, "dy": dy, "dw1": dw1, "db1": db1,
                "dx": rstd[:, None] * g * (dy - c1 - xhat * c2), "dgamma": (dy * xhat).sum(0), "dbeta": dy.sum(0)}
    if op == "resnet_block":
        w = {n: t["w" + n] * t["w" + n + "_scale"][:, None, None, None] if case["weights"] == "int8" else t["w" + n]
             for n in "123"}
        c1 = _conv64(t["x"], w["1"], t["b1"], 1, 0).relu()
        c2 = _conv64(c1, w["2"], t["b2"], case["s"], 1).relu()
        return {"c1": c1, "c2": c2, "c3": _conv64(c2, w["3"], t["b3"], 1, 0)}
    if op == "conv_train":
        x, w = t["x"].requires_grad_(), t["w"].requires_grad_()
        y = _conv64(x, w, None, case["s"], case["k"] // 2)
        dx, dw = torch.autograd.grad(y, (x, w), t["dy"])
        return {"y": y.detach(), "dx": dx, "dw": dw}
    if op.startswith("w8a16"):
        h = F.silu(t["x"] @ (t["up"] * t["up_scale"][:, None]).T.contiguous())
        return {"h": h, "y": h @ (t["down"] * t["down_scale"][:, None]).T.contiguous()}
    dx, dw, db = _linear_grads64(t["x"], t["w"], t["dy"])
    return {"y": t["x"] @ t["w"].T.contiguous() + t["b"], "dx": dx, "dw": dw, "db": db}
