"""The work that a user of this framework has it do, as cases that can be timed and checked.

Each case goes through public entry points: the packed layers (``modules``), the codec and the
nearest-centre assignment (``ops``), the QAT functions (``qat``) and two whole models
(``bench_models``).  ``listed()`` names twelve cases, ``draw()`` gives more of the same ranges,
``exact()`` computes a case's results in 64 bits with plain torch.

Weights come as what a packed checkpoint holds: a b-bit index stream and a codebook.  The indices
are uniform, as a quantile codebook makes them; the codebooks are sorted normal quantiles times a
scale per row.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

DEV = "cuda"
DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"fp32": 4, "fp16": 2, "bf16": 2}
PATCH, IMAGE, DIM, HEADS, DEPTH, MLP, CLASSES = 16, 224, 768, 12, 12, 3072, 1000


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def _linear(name, m, n, k, bits, dtype, out, per_channel=True, bias=True, act="none", residual="none", centers=0):
    c = dict(kind="linear", m=m, n=n, k=k, bits=bits, dtype=dtype, out=out, per_channel=per_channel, bias=bias,
             act=act, residual=residual, centers=centers)
    return dict(name=name, **c) if name else c


def _conv(name, b, c, h, w, oc, ks, stride, pad, bits, dtype, out, nhwc, per_channel=True, bias=True, act="none",
          residual=False, groups=1, dil=1):
    d = dict(kind="conv", b=b, c=c, h=h, w=w, oc=oc, ks=ks, stride=stride, pad=pad, bits=bits, dtype=dtype, out=out,
             nhwc=nhwc, per_channel=per_channel, bias=bias, act=act, residual=residual, groups=groups, dil=dil)
    return dict(name=name, **d) if name else d


def listed():
    return [
        # one token through a square decoder projection: the smallest call there is, a weight stream
        _linear("decode_token", 1, 4096, 4096, 3, "bf16", "bf16", bias=False),
        # a few sequences at once through a layer whose sizes fit no tile
        _linear("decode_ragged", 7, 4607, 1536, 4, "fp16", "fp16", per_channel=False),
        # one 224x224 image's tokens through the first MLP layer, GELU fused: latency of a single request
        _linear("linear_one_image", 197, 3072, 768, 4, "bf16", "fp16", act="gelu"),
        # a batch of 64 images through the second MLP layer with its residual: throughput
        _linear("linear_batch", 64 * 197, 768, 3072, 4, "fp16", "bf16", residual="bf16"),
        # the reference's own W4A4 Linear (float activations in, u4 codes inside), eight images
        dict(name="w4a4_linear", kind="lut_linear", m=8 * 197, n=3072, k=768, dtype="fp32", codebook="fp16", zp=7,
             scale=0.2371, bias=True),
        # the reference's own W4A4 Conv2d on NCHW floats: a late 3x3 layer of a residual network
        dict(name="w4a4_conv", kind="lut_conv", b=32, c=256, h=14, w=14, oc=256, ks=3, stride=1, pad=1, dtype="fp32",
             codebook="fp16", zp=0, scale=0.25, bias=True, groups=1),
        # weight-only 3x3 convolution in the reference's memory order, fp32 results
        _conv("conv_nchw", 32, 64, 56, 56, 64, 3, 1, 1, 2, "fp16", "fp32", False, bias=False),
        # a strided layer of a small serving batch, channels last as inside a network
        _conv("conv_serving", 8, 128, 28, 28, 256, 3, 2, 1, 2, "fp16", "fp16", True, act="relu"),
        # a quantization-aware training step's work on one weight: fake quantization, both regularizers, gradients
        dict(name="qat_layer", kind="qat", n=512 * 512 * 9, centers=16, dtype="fp32", tau=1e-4, soft=True, sigma=0.02),
        # export and load of one layer: nearest centres, packing, unpacking
        dict(name="codec_layer", kind="codec", rows=4096, cols=4096, bits=3, per_channel=True, dtype="fp32"),
        # whole models: a serving batch, and a throughput batch
        dict(name="resnet18_b16", kind="resnet18", b=16),
        dict(name="vit_b16_b64", kind="vit", b=64),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_linear(rng):
    bits = rng.choice((2, 3, 4, 4, 8))
    if rng.random() < 0.6:  # the widths of real layers
        n, k = rng.choice((192, 512, 768, 1000, 2304, 3072, 4096)), rng.choice((384, 512, 768, 1024, 2048, 3072, 4096))
    else:  # any width
        n, k = _log(rng, 33, 4608), _log(rng, 33, 4608)
    m = _log(rng, 1, min(12608, int(3.0e10 / (2 * n * k)) + 1))
    dtype = rng.choice(("bf16", "fp16", "fp32"))
    if rng.random() < 0.1:  # a layer trained with an activation codebook
        return _linear(None, m, n, k, bits, dtype, dtype, centers=rng.choice((16, 64)), bias=rng.random() < 0.5)
    out = dtype if rng.random() < 0.6 else rng.choice(("bf16", "fp16", "fp32"))
    act = rng.choice(("none", "none", "gelu", "relu"))
    residual = rng.choice(("none", out)) if act != "gelu" else "none"
    return _linear(None, m, n, k, bits, dtype, out, rng.random() < 0.7, rng.random() < 0.7, act, residual)


def _conv_size(rng):
    """A layer of a residual network, or any convolution, of at most about 8 GFLOP."""
    if rng.random() < 0.6:
        c = rng.choice((64, 64, 128, 256, 512))
        h = w = {64: 56, 128: 28, 256: 14, 512: 7}[c]
        oc, ks, stride = rng.choice(((c, 3, 1), (c, 3, 1), (2 * c, 3, 2), (2 * c, 1, 2)))
    else:
        c, oc = rng.choice((3, 16, 24, 48, 96, 100, 192, 320)), rng.choice((8, 30, 64, 96, 130, 256))
        h, w = _log(rng, 5, 80), _log(rng, 5, 80)
        ks, stride = rng.choice(((3, 1), (3, 2), (1, 1), (5, 1), (7, 2)))
    pad = ks // 2
    oh, ow = (h + 2 * pad - ks) // stride + 1, (w + 2 * pad - ks) // stride + 1
    b = _log(rng, 1, max(1, min(128, int(8e9 / (2 * c * oc * ks * ks * oh * ow)))))
    return b, c, h, w, oc, ks, stride, pad


def draw(rng):
    kind = rng.choice(("linear",) * 5 + ("conv",) * 4 + ("lut_linear", "lut_conv", "qat", "codec", "resnet18", "vit"))
    if kind == "linear":
        return _draw_linear(rng)
    if kind == "conv":
        b, c, h, w, oc, ks, stride, pad = _conv_size(rng)
        dtype = rng.choice(("fp16", "fp16", "fp16", "bf16", "fp32"))
        act = rng.choice(("none", "relu"))
        groups = 2 if c % 2 == 0 and oc % 2 == 0 and rng.random() < 0.1 else 1
        dil = 2 if ks == 3 and stride == 1 and min(h, w) > 6 and rng.random() < 0.1 else 1
        return _conv(None, b, c, h, w, oc, ks, stride, pad * dil, rng.choice((2, 2, 3, 4, 8)), dtype,
                     dtype if rng.random() < 0.7 else "fp32", rng.random() < 0.6, rng.random() < 0.8,
                     rng.random() < 0.8, act, act == "relu" and rng.random() < 0.5, groups, dil)
    if kind == "lut_linear":
        n, k = rng.choice(((3072, 768), (768, 3072), (1000, 512), (_log(rng, 33, 4096), _log(rng, 33, 4096))))
        return dict(kind=kind, m=_log(rng, 1, min(8192, int(2.0e10 / (2 * n * k)) + 1)), n=n, k=k,
                    dtype=rng.choice(("fp32", "fp32", "fp16", "bf16")), codebook=rng.choice(("fp16", "fp16", "fp32")),
                    zp=rng.choice((0, 7, 8)), scale=rng.choice((0.2371, 0.25, 0.2)), bias=rng.random() < 0.7)
    if kind == "lut_conv":
        b, c, h, w, oc, ks, stride, pad = _conv_size(rng)
        groups = 2 if c % 2 == 0 and oc % 2 == 0 and rng.random() < 0.1 else 1
        return dict(kind=kind, b=b, c=c, h=h, w=w, oc=oc, ks=ks, stride=stride, pad=pad,
                    dtype=rng.choice(("fp32", "fp32", "fp16")), codebook=rng.choice(("fp16", "fp16", "fp32")),
                    zp=rng.choice((0, 7)), scale=rng.choice((0.2371, 0.25)), bias=rng.random() < 0.7, groups=groups)
    if kind == "qat":
        centers = rng.choice((4, 8, 16, 16, 256))
        return dict(kind=kind, n=_log(rng, 500, 2400000 if centers <= 16 else 600000), centers=centers,
                    dtype=rng.choice(("fp32", "fp32", "bf16")), tau=rng.choice((1e-2, 1e-3, 1e-4, 1e-5)),
                    soft=rng.random() < 0.5, sigma=rng.choice((0.02, 0.05)))
    if kind == "codec":
        return dict(kind=kind, rows=_log(rng, 16, 4096), cols=_log(rng, 27, 4608), bits=rng.choice((2, 3, 4, 8)),
                    per_channel=rng.random() < 0.5, dtype=rng.choice(("fp32", "fp32", "bf16")))
    return dict(kind=kind, b=_log(rng, 1, 128 if kind == "resnet18" else 64))


# ---------------------------------------------------------------------------
# inputs, made from the seed alone
# ---------------------------------------------------------------------------

def _gen(case, seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + 17)


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _codebook(g, rows, size, scale):
    """[rows, size] sorted normal quantiles, each row with its own spread, entries jittered."""
    q = torch.linspace(0.0, 1.0, size + 2, device=DEV)[1:-1]
    base = math.sqrt(2.0) * torch.erfinv(2.0 * q - 1.0)
    spread = scale * (1.0 + 0.2 * torch.rand(rows, 1, device=DEV, generator=g))
    return ((base + 0.02 * _randn(g, rows, size)) * spread).sort(dim=1).values.contiguous()


def _indices(g, n, k, bits):
    return torch.randint(0, 1 << bits, (n, k), device=DEV, generator=g, dtype=torch.uint8)


def _pack(idx, bits):
    """LSB-first b-bit stream of the indices: what a packed checkpoint holds."""
    flat = idx.reshape(-1)
    if bits == 8:
        return flat.clone()
    if bits == 3:
        flat = F.pad(flat, (0, -flat.numel() % 8)).view(-1, 8).int()
        word = (flat << torch.arange(0, 24, 3, device=DEV, dtype=torch.int32)).sum(1, dtype=torch.int32)
        out = torch.stack([word & 255, (word >> 8) & 255, word >> 16], 1).to(torch.uint8).reshape(-1)
    else:
        per = 8 // bits
        flat = F.pad(flat, (0, -flat.numel() % per)).view(-1, per)
        out = (flat << torch.arange(0, 8, bits, device=DEV, dtype=torch.uint8)).sum(1, dtype=torch.uint8)
    return out[: (idx.numel() * bits + 7) // 8].contiguous()


def _weight(g, n, k, bits, per_channel, fan_in=None):
    """(indices, codebook) of a layer with n rows of k weights."""
    idx = _indices(g, n, k, bits)
    cb = _codebook(g, n if per_channel else 1, 1 << bits, 1.0 / math.sqrt(fan_in or k))
    return idx, cb


def _dequant(idx, cb):
    return torch.gather(cb.double().expand(idx.shape[0], -1), 1, idx.long())


def _linear_inputs(c, seed):
    g = _gen(c, seed)
    idx, cb = _weight(g, c["n"], c["k"], c["bits"], c["per_channel"])
    d = {"idx": idx, "cb": cb, "x": _randn(g, c["m"], c["k"]).to(DT[c["dtype"]])}
    d["bias"] = 0.1 * _randn(g, c["n"]) if c["bias"] else None
    d["res"] = _randn(g, c["m"], c["n"]).to(DT[c["residual"]]) if c["residual"] != "none" else None
    d["centers"] = _codebook(g, 1, c["centers"], 1.0)[0] if c["centers"] else None
    return d


def _conv_inputs(c, seed):
    g = _gen(c, seed)
    k = c["c"] // c["groups"] * c["ks"] ** 2
    idx, cb = _weight(g, c["oc"], k, c["bits"], c["per_channel"])
    x = torch.relu(_randn(g, c["b"], c["c"], c["h"], c["w"])).to(DT[c["dtype"]])
    d = {"idx": idx, "cb": cb, "x": x, "bias": 0.1 * _randn(g, c["oc"]) if c["bias"] else None}
    oh, ow = _out_hw(c)
    d["res"] = _randn(g, c["b"], c["oc"], oh, ow).to(DT[c["out"]]) if c["residual"] else None
    return d


def _lut_inputs(c, seed):
    g = _gen(c, seed)
    conv = c["kind"] == "lut_conv"
    n, k = (c["oc"], c["c"] // c["groups"] * c["ks"] ** 2) if conv else (c["n"], c["k"])
    idx, cb = _weight(g, n, k, 4, False)
    x = _randn(g, c["b"], c["c"], c["h"], c["w"]) if conv else _randn(g, c["m"], c["k"])
    x = torch.relu(x) if c["zp"] == 0 else x
    return {"idx": idx, "cb": cb[0].to(DT[c["codebook"]]), "x": x.to(DT[c["dtype"]]),
            "bias": 0.1 * _randn(g, n) if c["bias"] else None}


def _out_hw(c):
    span = c.get("dil", 1) * (c["ks"] - 1) + 1
    return (c["h"] + 2 * c["pad"] - span) // c["stride"] + 1, (c["w"] + 2 * c["pad"] - span) // c["stride"] + 1


def _qat_inputs(c, seed):
    g = _gen(c, seed)
    w = (c["sigma"] * _randn(g, c["n"])).to(DT[c["dtype"]])
    return {"w": w, "centers": _codebook(g, 1, c["centers"], c["sigma"])[0], "grad": _randn(g, c["n"]).to(w.dtype)}


def _codec_inputs(c, seed):
    g = _gen(c, seed)
    w = (_randn(g, c["rows"], c["cols"]) / math.sqrt(c["cols"])).to(DT[c["dtype"]])
    cb = _codebook(g, c["rows"] if c["per_channel"] else 1, 1 << c["bits"], 1.0 / math.sqrt(c["cols"]))
    return {"w": w, "cb": cb if c["per_channel"] else cb[0]}


# the layers of the two models, as (name, rows, weights per row, bits)
def _resnet_layers():
    layers = [("conv1", (64, 3, 7, 7), 2, 3, 8)]
    cin = 64
    for i, cout in enumerate((64, 128, 256, 512)):
        for j in range(2):
            stride = 2 if i and not j else 1
            p = f"layer{i + 1}.{j}."
            layers.append((p + "conv1", (cout, cin, 3, 3), stride, 1, 2))
            layers.append((p + "conv2", (cout, cout, 3, 3), 1, 1, 2))
            if stride == 2:
                layers.append((p + "downsample", (cout, cin, 1, 1), stride, 0, 4))
            cin = cout
    return layers


def _resnet_inputs(c, seed):
    g = _gen(c, seed)
    d = {"x": _randn(g, c["b"], 3, IMAGE, IMAGE).half()}
    for name, (oc, ic, kh, kw), _, _, bits in _resnet_layers():
        # sqrt(2 / fan-in) keeps the activations' size from layer to layer; the second conv of a block is damped
        scale = 2.0 * (ic * kh * kw) if name.endswith("conv2") else 0.5 * (ic * kh * kw)
        idx, cb = _weight(g, oc, ic * kh * kw, bits, True, scale)
        d[name] = (idx, cb, 0.1 * _randn(g, oc))
    idx, cb = _weight(g, CLASSES, 512, 8, True)
    d["fc"] = (idx, cb, 0.05 * _randn(g, CLASSES))
    return d


VIT_LINEARS = (("attn.qkv", 3 * DIM, DIM), ("attn.proj", DIM, DIM), ("fc1", MLP, DIM), ("fc2", DIM, MLP))


def _vit_inputs(c, seed):
    g = _gen(c, seed)
    bf = torch.bfloat16
    d = {"x": _randn(g, c["b"], 3, IMAGE, IMAGE).to(bf), "cls": (0.02 * _randn(g, 1, 1, DIM)).to(bf),
         "pos": (0.02 * _randn(g, 1, (IMAGE // PATCH) ** 2 + 1, DIM)).to(bf),
         "embed": ((_randn(g, DIM, 3 * PATCH * PATCH) / math.sqrt(3 * PATCH * PATCH)).to(bf),
                   (0.02 * _randn(g, DIM)).to(bf)),
         "head": ((0.02 * _randn(g, CLASSES, DIM)).to(bf), (0.02 * _randn(g, CLASSES)).to(bf))}
    norms = [f"blocks.{i}.{ln}" for i in range(DEPTH) for ln in ("ln_1", "ln_2")] + ["ln"]
    for name in norms:
        d[name] = ((1.0 + 0.1 * _randn(g, DIM)).to(bf), (0.05 * _randn(g, DIM)).to(bf))
    for i in range(DEPTH):
        for leaf, n, k in VIT_LINEARS:
            idx, cb = _weight(g, n, k, 4, True, 1.0 / 0.02 ** 2)  # weights of size 0.02
            d[f"blocks.{i}.{leaf}"] = (idx, cb, 0.02 * _randn(g, n))
    return d


# ---------------------------------------------------------------------------
# what a program has in hand before the call
# ---------------------------------------------------------------------------

def _set(model, name, new):
    parent, _, leaf = name.rpartition(".")
    setattr(model.get_submodule(parent) if parent else model, leaf, new)


def _resnet_state(c, seed):
    from dimq_amd.bench_models import ResNet18
    from dimq_amd.modules import DIMQCodebookConv2d, DIMQCodebookLinear, DIMQMaxPool2d
    d = _resnet_inputs(c, seed)
    with torch.device("meta"):
        model = ResNet18(CLASSES)
    for name, shape, stride, pad, bits in _resnet_layers():
        idx, cb, bias = d[name]
        _set(model, name, DIMQCodebookConv2d(_pack(idx, bits), cb, bits, shape, bias, stride=stride, padding=pad,
                                             out_dtype=torch.float16))
    idx, cb, bias = d["fc"]
    model.fc = DIMQCodebookLinear(_pack(idx, 8), cb, 8, CLASSES, 512, bias, out_dtype=torch.float16)
    model.maxpool = DIMQMaxPool2d.from_max_pool(model.maxpool)
    return {"model": model.eval(), "x": d["x"].contiguous(memory_format=torch.channels_last)}


def _vit_state(c, seed):
    from dimq_amd.bench_models import ViT
    from dimq_amd.modules import DIMQCodebookLinear, DIMQLayerNorm
    d = _vit_inputs(c, seed)
    with torch.device("meta"):
        model = ViT()
    frozen = lambda t: torch.nn.Parameter(t, requires_grad=False)  # noqa: E731
    for i in range(DEPTH):
        for leaf, n, k in VIT_LINEARS:
            name = f"blocks.{i}.{leaf}"
            idx, cb, bias = d[name]
            # tensors that only feed another codebook layer or attention are written in fp16
            out = torch.float16 if leaf in ("attn.qkv", "fc1") else torch.bfloat16
            _set(model, name, DIMQCodebookLinear(_pack(idx, 4), cb, 4, n, k, bias, out_dtype=out))
    for name in [k for k in d if k.rsplit(".", 1)[-1] in ("ln", "ln_1", "ln_2")]:
        ln = torch.nn.LayerNorm(DIM, eps=1e-6, device=DEV, dtype=torch.bfloat16)
        ln.weight, ln.bias = frozen(d[name][0]), frozen(d[name][1])
        new = DIMQLayerNorm.from_layer_norm(ln, None if name == "ln" else torch.float16)
        _set(model, name, new.requires_grad_(False))
    model.class_token, model.pos_embedding = frozen(d["cls"]), frozen(d["pos"])
    model.conv_proj.weight = frozen(d["embed"][0].view(DIM, 3, PATCH, PATCH))
    model.conv_proj.bias = frozen(d["embed"][1])
    model.head.weight, model.head.bias = frozen(d["head"][0]), frozen(d["head"][1])
    return {"model": model.eval(), "x": d["x"]}


def prepare(case, seed):
    from dimq_amd import modules
    c, kind = case, case["kind"]
    if kind in ("resnet18", "vit"):
        s = _resnet_state(c, seed) if kind == "resnet18" else _vit_state(c, seed)
        return {"kind": kind, **s}
    if kind == "linear":
        d = _linear_inputs(c, seed)
        layer = modules.DIMQCodebookLinear(_pack(d["idx"], c["bits"]), d["cb"], c["bits"], c["n"], c["k"], d["bias"],
                                           out_dtype=DT[c["out"]], activation_centers=d["centers"])
        return {"kind": kind, "layer": layer, "x": d["x"], "res": d["res"], "act": None if c["act"] == "none" else c["act"]}
    if kind == "conv":
        d = _conv_inputs(c, seed)
        layer = modules.DIMQCodebookConv2d(
            _pack(d["idx"], c["bits"]), d["cb"], c["bits"], (c["oc"], c["c"] // c["groups"], c["ks"], c["ks"]),
            d["bias"], stride=c["stride"], padding=c["pad"], dilation=c["dil"], groups=c["groups"],
            out_dtype=DT[c["out"]])
        mf = torch.channels_last if c["nhwc"] else torch.contiguous_format
        res = None if d["res"] is None else d["res"].contiguous(memory_format=mf)
        return {"kind": "conv", "layer": layer, "x": d["x"].contiguous(memory_format=mf), "res": res,
                "act": None if c["act"] == "none" else c["act"]}
    if kind == "lut_linear":
        d = _lut_inputs(c, seed)
        return {"kind": kind, "x": d["x"], "layer": modules.DIMQLinear(
            _pack(d["idx"], 4), d["cb"], c["scale"], c["zp"], c["n"], c["k"], d["bias"])}
    if kind == "lut_conv":
        d = _lut_inputs(c, seed)
        return {"kind": kind, "x": d["x"], "layer": modules.DIMQConv2d(
            _pack(d["idx"], 4), d["cb"], c["scale"], c["zp"], (c["oc"], c["c"] // c["groups"], c["ks"], c["ks"]),
            d["bias"], stride=c["stride"], padding=c["pad"], groups=c["groups"])}
    if kind == "qat":
        d = _qat_inputs(c, seed)
        return {"kind": kind, "w": d["w"].requires_grad_(), "centers": d["centers"].requires_grad_(),
                "grad": d["grad"], "tau": c["tau"], "soft": c["soft"],
                "weights": (torch.tensor(0.5, device=DEV), torch.tensor(2.0, device=DEV))}
    d = _codec_inputs(c, seed)
    return {"kind": kind, "w": d["w"], "cb": d["cb"], "bits": c["bits"], "per_channel": c["per_channel"]}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind in ("linear", "conv"):
        with torch.no_grad():
            if state["res"] is None and state["act"] is None:
                return state["layer"](state["x"])
            return state["layer"](state["x"], residual=state["res"], activation=state["act"])
    if kind in ("lut_linear", "lut_conv"):
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "qat":
        from dimq_amd import qat
        w, c = state["w"], state["centers"]
        wq = qat.soft_dequantize_weight(w, c, state["tau"]) if state["soft"] else qat.fake_quant_weight_ste(w, c)
        softmin = qat.dimq_softmin_loss(w, c, state["tau"])
        separation = qat.separation_loss(w, c)
        gw, gc = torch.autograd.grad((wq, softmin, separation), (w, c), (state["grad"], *state["weights"]))
        return {"wq": wq, "softmin": softmin, "separation": separation, "grad_w": gw, "grad_c": gc}
    if kind == "codec":
        from dimq_amd import ops
        idx, values = ops.hard_quantize(state["w"], state["cb"], state["per_channel"])
        packed = ops.pack_bits(idx, state["bits"])
        return {"idx": idx, "values": values, "packed": packed,
                "unpacked": ops.unpack_bits(packed, idx.numel(), state["bits"])}
    with torch.no_grad():
        return state["model"](state["x"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    if kind in ("linear", "lut_linear"):
        m, n, k = c["m"], c["n"], c["k"]
        bits = c.get("bits", 4)
        by = m * k * SIZE[c["dtype"]] + n * k * bits // 8 + m * n * SIZE[c.get("out", "fp32")] + 4 * n * c["bias"]
        by += (n if c.get("per_channel") else 1) * (1 << bits) * 4
        if c.get("residual", "none") != "none":
            by += m * n * SIZE[c["residual"]]
        return {"bytes": by, "flops": 2 * m * n * k}
    if kind in ("conv", "lut_conv"):
        oh, ow = _out_hw(c)
        bits, k = c.get("bits", 4), c["c"] // c["groups"] * c["ks"] ** 2
        out = c["b"] * c["oc"] * oh * ow
        by = c["b"] * c["c"] * c["h"] * c["w"] * SIZE[c["dtype"]] + c["oc"] * k * bits // 8
        by += out * SIZE[c.get("out", "fp32")] * (2 if c.get("residual") else 1)
        return {"bytes": by, "flops": 2 * out * k}
    if kind == "qat":
        # w and the incoming gradient in, the quantized weight and its gradient out; a difference, a square, an
        # exponential and two sums per weight and centre, of each of the two functions in each direction
        return {"bytes": 4 * c["n"] * SIZE[c["dtype"]], "flops": c["n"] * c["centers"] * 6 * (4 if c["soft"] else 2)}
    if kind == "codec":
        n, s = c["rows"] * c["cols"], SIZE[c["dtype"]]
        return {"bytes": n * (2 * s + 2) + n * c["bits"] // 8, "flops": 3 * n * c["bits"]}
    if kind == "resnet18":
        flops, hw = 0, {"conv1": 112}
        for name, (oc, ic, kh, kw), *_ in _resnet_layers():
            side = 112 if name == "conv1" else 56 >> (int(name[5]) - 1)
            flops += 2 * side * side * oc * ic * kh * kw
        weights = sum(oc * ic * kh * kw * bits // 8 for _, (oc, ic, kh, kw), _, _, bits in _resnet_layers())
        return {"bytes": c["b"] * (3 * IMAGE * IMAGE + CLASSES) * 2 + weights + CLASSES * 512,
                "flops": c["b"] * (flops + 2 * 512 * CLASSES)}
    tok = (IMAGE // PATCH) ** 2 + 1
    layer = sum(2 * n * k for _, n, k in VIT_LINEARS) * tok + 4 * tok * tok * DIM
    flops = c["b"] * (DEPTH * layer + 2 * (tok - 1) * DIM * 3 * PATCH * PATCH + 2 * DIM * CLASSES)
    weights = DEPTH * sum(n * k // 2 + 64 * n for _, n, k in VIT_LINEARS) + 2 * DIM * (3 * PATCH * PATCH + CLASSES)
    return {"bytes": c["b"] * (3 * IMAGE * IMAGE + CLASSES) * 2 + weights, "flops": flops}


def tolerance(case):
    # about four times the error against 64 bits that a hundred drawn cases showed
    kind = case["kind"]
    if kind == "codec":
        return "exact"
    if kind == "linear":  # fp16 weights and activations at the matrix cores, one rounding of the result
        return {"rel": {"fp32": 1.5e-3, "fp16": 1.5e-3, "bf16": 7e-3}[case["out"]]}
    if kind == "conv":  # few distinct weights, so that the rounding of one entry repeats in every product
        return {"rel": {"fp32": 8e-3, "fp16": 7e-3, "bf16": 9e-3}[case["out"]]}
    if kind in ("lut_linear", "lut_conv"):
        return {"rel": 3e-6}  # 32-bit sums of exact codes and fp32 products
    if kind == "qat":
        return {"rel": 7e-6 if case["dtype"] == "fp32" else 9e-3}
    return {"rel": 3e-2 if kind == "vit" else 1e-2}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------

def _conv64(x, w, bias, stride, pad, dil=1, groups=1):
    """2-d convolution as products of unfolded patches, a few images at a time."""
    b, c, h, wd = x.shape
    oc, icg, kh, kw = w.shape
    oh, ow = (h + 2 * pad - dil * (kh - 1) - 1) // stride + 1, (wd + 2 * pad - dil * (kw - 1) - 1) // stride + 1
    w2 = w.reshape(groups, oc // groups, icg * kh * kw)
    y = torch.empty(b, oc, oh * ow, dtype=torch.float64, device=x.device)
    step = max(1, int(2.5e7 / (c * kh * kw * oh * ow)))
    for i in range(0, b, step):
        u = F.unfold(x[i:i + step], (kh, kw), dilation=dil, padding=pad, stride=stride)
        u = u.view(u.shape[0], groups, icg * kh * kw, oh * ow)
        for q in range(groups):
            lo, hi = q * (oc // groups), (q + 1) * (oc // groups)
            y[i:i + step, lo:hi] = torch.matmul(w2[q], u[:, q])
    y = y.view(b, oc, oh, ow)
    return y if bias is None else y + bias.double().view(1, -1, 1, 1)


def _post64(y, res, act):
    if res is not None:
        y = y + res.double()
    return torch.relu(y) if act == "relu" else F.gelu(y) if act == "gelu" else y


def _u4_64(x, scale, zp):
    """The activations that the u4 codes stand for: codes by a 32-bit division, as the format says."""
    q = x.float() / torch.tensor(scale, dtype=torch.float32, device=x.device)
    return ((torch.round(q) + zp).clamp(0, 15).double() - zp) * scale


def _nearest(x, centers):
    """Index of the first nearest centre, by 32-bit squared distances."""
    flat, out = x.reshape(-1).float(), []
    for part in flat.split(1 << 20):
        out.append((part[:, None] - centers[None, :]).square().argmin(1))
    return torch.cat(out).view(x.shape)


def _qat64(c, seed):
    d = _qat_inputs(c, seed)
    w, cs, tau, n = d["w"].double(), d["centers"].double(), c["tau"], c["n"]
    wq, gw, gc, softmin = torch.empty_like(w), torch.empty_like(w), torch.zeros_like(cs), 0.0
    up = d["grad"].double()
    for i in range(0, n, 1 << 18):
        s = slice(i, i + (1 << 18))
        diff = w[s, None] - cs[None, :]
        z = -diff.square() / tau
        p = torch.softmax(z, 1)
        softmin += float((-tau * (torch.logsumexp(z, 1) - math.log(c["centers"]))).sum())
        gw[s] = 0.5 * (p * 2 * diff).sum(1)
        gc += -0.5 * 2 * (p * diff).sum(0)
        if c["soft"]:
            out = p @ cs
            wq[s] = out
            slope = p * (cs - out[:, None]) * (2 / tau)
            gw[s] += up[s] * (-slope * diff).sum(1)
            gc += (up[s, None] * (p + slope * diff)).sum(0)
        else:
            wq[s] = cs[(w[s, None].float() - d["centers"][None, :]).square().argmin(1)]
            gw[s] += up[s]
    delta = 6.0 * w.std(unbiased=False) / c["centers"]
    gap = cs[:, None] - cs[None, :]
    r = torch.sqrt(gap.square() + 1e-12)
    hinge = torch.relu(delta - r)
    off = ~torch.eye(c["centers"], dtype=torch.bool, device=w.device)
    separation = 0.5 * hinge.square()[off].sum()
    gc += 2.0 * torch.where(off, -2.0 * hinge * gap / r, 0.0).sum(1)
    return {"wq": wq, "softmin": torch.tensor(softmin, dtype=torch.float64), "separation": separation, "grad_w": gw,
            "grad_c": gc}


def _resnet64(c, seed):
    d = _resnet_inputs(c, seed)

    def conv(name, x):
        shape, stride, pad = next((s, st, p) for n, s, st, p, _ in _resnet_layers() if n == name)
        idx, cb, bias = d[name]
        return _conv64(x, _dequant(idx, cb).view(shape), bias, stride, pad)

    x = F.max_pool2d(torch.relu(conv("conv1", d["x"].double())), 3, 2, 1)
    for i in range(1, 5):
        for j in range(2):
            p = f"layer{i}.{j}."
            y = conv(p + "conv2", torch.relu(conv(p + "conv1", x)))
            x = torch.relu(y + (conv(p + "downsample", x) if p + "downsample" in d else x))
    idx, cb, bias = d["fc"]
    return x.mean((2, 3)) @ _dequant(idx, cb).T + bias.double()


def _vit64(c, seed):
    d, b, p = _vit_inputs(c, seed), c["b"], PATCH
    side = IMAGE // p

    def linear(name, x):
        idx, cb, bias = d[name]
        return x @ _dequant(idx, cb).T + bias.double()

    def norm(name, x):
        return F.layer_norm(x, (DIM,), d[name][0].double(), d[name][1].double(), 1e-6)

    x = d["x"].double().view(b, 3, side, p, side, p).permute(0, 2, 4, 1, 3, 5).reshape(b, side * side, 3 * p * p)
    x = x @ d["embed"][0].double().T + d["embed"][1].double()
    x = torch.cat([d["cls"].double().expand(b, -1, -1), x], 1) + d["pos"].double()
    t = x.shape[1]
    for i in range(DEPTH):
        q, k, v = linear(f"blocks.{i}.attn.qkv", norm(f"blocks.{i}.ln_1", x)).view(b, t, 3, HEADS, -1).permute(2, 0, 3, 1, 4)
        a = torch.softmax(torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(DIM // HEADS), -1)
        x = x + linear(f"blocks.{i}.attn.proj", torch.matmul(a, v).transpose(1, 2).reshape(b, t, DIM))
        x = x + linear(f"blocks.{i}.fc2", F.gelu(linear(f"blocks.{i}.fc1", norm(f"blocks.{i}.ln_2", x))))
    return norm("ln", x[:, 0]) @ d["head"][0].double().T + d["head"][1].double()


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear":
        d = _linear_inputs(c, seed)
        x = d["x"].double()
        if c["centers"]:
            x = d["centers"].to(d["x"].dtype).double()[_nearest(d["x"], d["centers"])]
        y = x @ _dequant(d["idx"], d["cb"]).T
        return _post64(y if d["bias"] is None else y + d["bias"].double(), d["res"], c["act"])
    if kind in ("conv", "lut_conv"):
        d = _conv_inputs(c, seed) if kind == "conv" else _lut_inputs(c, seed)
        cb = d["cb"] if kind == "conv" else d["cb"][None, :]
        w = _dequant(d["idx"], cb).view(c["oc"], -1, c["ks"], c["ks"])
        x = d["x"].double() if kind == "conv" else _u4_64(d["x"], c["scale"], c["zp"])
        y = _conv64(x, w, d["bias"], c["stride"], c["pad"], c.get("dil", 1), c["groups"])
        return _post64(y, d.get("res"), c.get("act", "none"))
    if kind == "lut_linear":
        d = _lut_inputs(c, seed)
        y = _u4_64(d["x"], c["scale"], c["zp"]) @ _dequant(d["idx"], d["cb"][None, :]).T
        return y if d["bias"] is None else y + d["bias"].double()
    if kind == "qat":
        return _qat64(c, seed)
    if kind == "codec":
        return None
    return _resnet64(c, seed) if kind == "resnet18" else _vit64(c, seed)
