"""The work that users of the phase-quantized layers have them do, as cases to time and to compare.

A case is one call of a public entry point with inputs of a stated size: a
whole model, one encoder block, one layer in inference, one training step of
a layer, the gradient through a frozen layer, or the single-plane primitive.
Weights are phase codes with per-row magnitudes (what an exported bundle
holds) or, in training, the float32 master weight; inputs are unit normal,
as behind a LayerNorm.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "rpfq-review_amd"))

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
DEV = "cuda"

# codebook -> (planes per U / W, bits per code)
BOOKS = {"axis1": (1, 2), "axis2": (2, 2), "sign2": (2, 2), "psk16": (1, 4), "table": (1, 4)}


def listed():
    return [
        # the flagship: one ViT-B/16 batch of 256 images through the packed
        # model in fp16, weights quantized, activations as they are
        {"name": "vit_b16_forward", "kind": "model", "model": "vit", "dim": 768, "heads": 12, "depth": 12,
         "batch": 256, "img": 224, "dtype": "fp16", "book": "axis2"},
        # the smallest model of the family at a serving batch: many short launches
        {"name": "deit_ti_forward", "kind": "model", "model": "deit", "dim": 192, "heads": 3, "depth": 12,
         "batch": 64, "img": 224, "dtype": "fp16", "book": "axis2"},
        # one image: an encoder block is a handful of launches of few rows
        {"name": "vit_b16_block_1img", "kind": "block", "dim": 768, "heads": 12, "batch": 1, "tokens": 197,
         "dtype": "fp16", "book": "axis2", "bits": 0, "rotate": False},
        # a bf16 model's block at a throughput batch
        {"name": "vit_b16_block_bf16", "kind": "block", "dim": 768, "heads": 12, "batch": 128, "tokens": 197,
         "dtype": "bf16", "book": "axis2", "bits": 0, "rotate": False},
        # validation as the training configuration runs it: float32, 4-bit
        # activations, rotated weights, 64 images (a layer and not a block:
        # 4-bit levels that tip in one layer move the next one's by 3%)
        {"name": "vit_b16_fc1_a4_f32", "kind": "layer", "rows": 64 * 197, "inf": 768, "outf": 3072, "dtype": "fp32",
         "book": "axis2", "bits": 4, "rotate": True},
        # the largest layer of the 16-PSK ViT-L/16 model, 64 images
        {"name": "vit_l16_fc1_psk16", "kind": "layer", "rows": 64 * 197, "inf": 1024, "outf": 4096, "dtype": "fp16",
         "book": "psk16", "bits": 0, "rotate": False},
        # Swin-T's first stage: a small layer over very many rows (128 images)
        {"name": "swin_t_stage0_qkv", "kind": "layer", "rows": 128 * 56 * 56, "inf": 96, "outf": 288, "dtype": "fp16",
         "book": "axis2", "bits": 0, "rotate": False},
        # the classifier of one image: a single row against all its codes
        {"name": "head_1img", "kind": "layer", "rows": 1, "inf": 768, "outf": 1000, "dtype": "fp16", "book": "axis2",
         "bits": 0, "rotate": False},
        # quantization-aware training of ViT-B/16 as the reference trains it:
        # float32, 64 images on a GPU, 4-bit activations; forward and backward
        {"name": "train_vit_b16_fc1", "kind": "train", "rows": 64 * 197, "inf": 768, "outf": 3072, "amp": False,
         "method": "complex_phase_v2", "bits": 4, "rotate": False},
        # the same under fp16 autocast
        {"name": "train_vit_b16_qkv_amp", "kind": "train", "rows": 64 * 197, "inf": 768, "outf": 2304, "amp": True,
         "method": "complex_phase_v2", "bits": 4, "rotate": False},
        # a frozen quantized layer inside a model that is tuned around it:
        # its output and the gradient that passes through it
        {"name": "frozen_vit_b16_fc2", "kind": "frozen", "rows": 64 * 197, "inf": 3072, "outf": 768, "dtype": "fp32",
         "book": "axis2", "bits": 0, "rotate": False},
        # the single-plane primitive at the ViT-B fc1 shape, 8 images
        {"name": "plane_vit_b16_fc1", "kind": "plane", "rows": 1576, "inf": 768, "outf": 3072, "block": 0,
         "conj": False},
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------
def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rows(rng, lo, hi, per_row, most):
    """A number of rows spread over its logarithm, at most `most` operations."""
    return _log_int(rng, lo, max(lo, min(hi, int(most // per_row))))


def _features(rng):
    """(in, out) of a layer: those of the model family's layers, or generic ones."""
    if rng.random() < 0.6:
        dim = rng.choice([96, 192, 384, 768, 1024])
        return rng.choice([(dim, 3 * dim), (dim, dim), (dim, 4 * dim), (4 * dim, dim), (dim, 1000), (2 * dim, dim)])
    return 16 * _log_int(rng, 3, 256), 2 * _log_int(rng, 24, 2048)


def draw(rng):
    kind = rng.choice(["block", "layer", "layer", "layer", "train", "train", "frozen", "plane"])
    if kind == "block":
        dim, heads = rng.choice([(192, 3), (384, 6), (768, 12), (1024, 16)])
        tokens = rng.choice([197, 198, 145, 257, 50 + rng.randrange(200)])
        per_image = 24 * tokens * dim * dim + 4 * tokens * tokens * dim
        return {"kind": "block", "dim": dim, "heads": heads, "batch": _rows(rng, 1, 256, per_image, 7e11),
                "tokens": tokens, "dtype": rng.choice(["fp16", "fp16", "bf16", "fp32"]),
                "book": rng.choice(["axis2", "axis2", "axis1", "sign2", "psk16"]), "bits": rng.choice([0, 0, 8]),
                "rotate": rng.random() < 0.3}
    if kind == "plane":
        inf, outf = 32 * _log_int(rng, 2, 64), _log_int(rng, 48, 4096)
        return {"kind": "plane", "rows": _rows(rng, 1, 50_000, 8 * inf * outf, 2.5e11), "inf": inf, "outf": outf,
                "block": rng.choice([0, 0, 32, 256]), "conj": rng.random() < 0.5}
    inf, outf = _features(rng)
    if kind == "train":
        return {"kind": "train", "rows": _rows(rng, 16, 50_000, 6 * inf * outf, 3e11), "inf": inf, "outf": outf,
                "amp": rng.random() < 0.35,
                "method": rng.choice(["complex_phase_v2", "complex_phase_v2", "complex_phase_v1", "complex_phase_v4",
                                      "complex_phase_new_v2"]),
                "bits": rng.choice([4, 4, 8, 0]), "rotate": rng.random() < 0.3}
    case = {"kind": kind, "inf": inf, "outf": outf, "dtype": rng.choice(["fp16", "fp16", "bf16", "fp32"]),
            "book": rng.choice(["axis2", "axis2", "axis1", "sign2", "psk16", "table"]),
            "bits": rng.choice([0, 0, 4, 8]), "rotate": False}
    case["rotate"] = case["book"] != "table" and rng.random() < 0.3
    passes = 2 if kind == "layer" else 4
    case["rows"] = _rows(rng, 1 if kind == "layer" else 16, 400_000, max(passes * inf * outf, 2000 * (inf + outf)), 6e11)
    return case


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * scale


def _codes(g, outf, inf, book, rotate):
    """One layer as an exported bundle holds it: code planes of U and W,
    their per-row scales (or value tables) and the rotation of each."""
    n, k = outf // 2, inf // 2
    per, bits = BOOKS[book]
    planes = [torch.randint(0, 256, (n, k * bits // 8), generator=g, device=DEV, dtype=torch.uint8)
              for _ in range(2 * per)]
    if book == "table":
        scales = [(_normal(g, n, 16, scale=0.02), _normal(g, n, 16, scale=0.02)) for _ in planes]
    else:  # coefficients of 0.02 to 0.03, as a trained layer has
        scales = [(s, s) for s in (0.003 + 0.027 * torch.rand(n, 1, generator=g, device=DEV) for _ in planes)]
    rotation = None
    if rotate:
        t = [float(v) for v in torch.randn(2, generator=torch.Generator().manual_seed(outf * 8192 + inf)) * 0.3]
        rotation = tuple(tuple(torch.tensor([math.cos(a), math.sin(a)], dtype=torch.float32).tolist()) for a in t)
    return {"n": n, "k": k, "book": book, "planes": planes, "scales": scales, "rotation": rotation,
            "bias": _normal(g, outf, scale=0.1)}


def _block_params(g, dim, book, rotate, dtype):
    p = {name: _codes(g, o, i, book, rotate) for name, o, i in
         (("qkv", 3 * dim, dim), ("proj", dim, dim), ("fc1", 4 * dim, dim), ("fc2", dim, 4 * dim))}
    for name in ("norm1", "norm2"):
        p[name] = _norm_params(g, dim, dtype)
    return p


def _norm_params(g, dim, dtype):
    return (1 + _normal(g, dim, scale=0.1)).to(dtype), _normal(g, dim, scale=0.1).to(dtype)


def _model_params(g, case):
    dtype, dim, prefix = DTYPES[case["dtype"]], case["dim"], 2 if case["model"] == "deit" else 1
    p = {"blocks": [_block_params(g, dim, case["book"], False, dtype) for _ in range(case["depth"])],
         "norm": _norm_params(g, dim, dtype),
         "heads": [_codes(g, 1000, dim, case["book"], False) for _ in range(prefix)],
         "patch": (_normal(g, dim, 3, 16, 16, scale=0.05).to(dtype), _normal(g, dim, scale=0.1).to(dtype)),
         "prefix": [_normal(g, 1, 1, dim, scale=0.5).to(dtype) for _ in range(prefix)],
         "pos": _normal(g, 1, (case["img"] // 16) ** 2 + prefix, dim, scale=0.3).to(dtype)}
    p["x"] = _normal(g, case["batch"], 3, case["img"], case["img"]).to(dtype)
    return p


def _train_params(g, case):
    p = {"weight": _normal(g, case["outf"], case["inf"], scale=0.02), "bias": _normal(g, case["outf"], scale=0.1),
         "x": _normal(g, case["rows"], case["inf"]), "gy": _normal(g, case["rows"], case["outf"], scale=0.1)}
    if case["amp"]:
        p["gy"] = p["gy"].half()
    p["angles"] = (0.2, -0.3) if case["rotate"] else None
    return p


def _plane_params(g, case):
    m, k, n, block = case["rows"], case["inf"], case["outf"], case["block"]
    nblk = 1 if block == 0 else -(-k // block)
    return {"xr": _normal(g, m, k), "xi": _normal(g, m, k),
            "codes": torch.randint(0, 256, (n, k // 4), generator=g, device=DEV, dtype=torch.uint8),
            "gamma": [(1.0 / (0.01 + 0.09 * torch.rand(n, nblk, generator=g, device=DEV))).half() for _ in range(2)]}


# ---------------------------------------------------------------------------
# what a program has in hand before the call
# ---------------------------------------------------------------------------
def _set_layer(layer, p):
    """Give a quantized layer its codes and bias, packed on the device."""
    from quant_models import _native as N
    from quant_models.packing import LayerCodes

    book = {"axis1": N.CB_AXIS, "axis2": N.CB_AXIS, "sign2": N.CB_SIGN, "psk16": N.CB_PSK16, "table": N.CB_TABLE}
    layer.load_packed(LayerCodes(p["planes"], [s[0] for s in p["scales"]], [s[1] for s in p["scales"]], p["n"], p["k"],
                                 book[p["book"]], BOOKS[p["book"]][0], 0, p["rotation"]))
    layer.bias.data = p["bias"].clone()
    layer.eval().packed(torch.device(DEV, torch.cuda.current_device()))


def _layer(case, p):
    from quant_models import QATLinearComplexPhase

    with torch.device(DEV):
        layer = QATLinearComplexPhase(enable_act_quant=case["bits"] > 0, act_num_bits=max(2, case["bits"]),
                                      in_features=case["inf"], out_features=case["outf"])
    _set_layer(layer, p)
    return layer


def _set_norm(norm, wb):
    norm.weight.data, norm.bias.data = wb[0].clone(), wb[1].clone()


def _set_block(block, p):
    for layer, name in ((block.attn.qkv, "qkv"), (block.attn.proj, "proj"), (block.mlp.fc1, "fc1"),
                        (block.mlp.fc2, "fc2")):
        _set_layer(layer, p[name])
    _set_norm(block.norm1, p["norm1"])
    _set_norm(block.norm2, p["norm2"])


def _build(case, dim, heads, depth, bits=0, img=224, cls="vit"):
    import contextlib
    import io

    from quant_models.quant_rpfq_deit import ComplexDeiT
    from quant_models.quant_rpfq_vit import ComplexVisionTransformer

    with torch.device(DEV), contextlib.redirect_stdout(io.StringIO()):
        model = (ComplexDeiT if cls == "deit" else ComplexVisionTransformer)(
            img_size=img, embed_dim=dim, depth=depth, num_heads=heads, norm_layer=torch.nn.LayerNorm,
            quant_method_u="complex_phase_v2", quant_method_w="complex_phase_v2", enable_act_quant=bits > 0,
            act_num_bits=max(2, bits), enable_rotation=False)
    for p in model.parameters():
        p.requires_grad_(False)
    return model


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "model":
        from quant_models.inference import prepare_inference

        p, dtype = _model_params(g, case), DTYPES[case["dtype"]]
        model = _build(case, case["dim"], case["heads"], case["depth"], img=case["img"], cls=case["model"])
        for block, b in zip(model.blocks, p["blocks"]):
            _set_block(block, b)
        _set_layer(model.head, p["heads"][0])
        model.cls_token.data = p["prefix"][0].clone()
        if case["model"] == "deit":
            _set_layer(model.head_dist, p["heads"][1])
            model.dist_token.data = p["prefix"][1].clone()
        _set_norm(model.norm, p["norm"])
        model.pos_embed.data = p["pos"].clone()
        model.patch_embed.proj.weight.data, model.patch_embed.proj.bias.data = (t.clone() for t in p["patch"])
        prepare_inference(model, DEV, dtype)
        return {"kind": kind, "f": model, "x": p["x"]}
    if kind == "block":
        from quant_models.inference import prepare_inference

        dtype = DTYPES[case["dtype"]]
        block = _build(case, case["dim"], case["heads"], 1, case["bits"], img=32).blocks[0]
        _set_block(block, _block_params(g, case["dim"], case["book"], case["rotate"], dtype))
        prepare_inference(block, DEV, dtype)
        return {"kind": kind, "f": block, "x": _normal(g, case["batch"], case["tokens"], case["dim"]).to(dtype)}
    if kind in ("layer", "frozen"):
        dtype = DTYPES[case["dtype"]]
        p = _codes(g, case["outf"], case["inf"], case["book"], case["rotate"])
        s = {"kind": kind, "f": _layer(case, p), "x": _normal(g, case["rows"], case["inf"]).to(dtype)}
        if kind == "frozen":
            for q in s["f"].parameters():
                q.requires_grad_(False)
            s["x"].requires_grad_(True)
            s["gy"] = _normal(g, case["rows"], case["outf"], scale=0.1).to(dtype)
        return s
    if kind == "train":
        from quant_models import QATLinearComplexPhase

        p = _train_params(g, case)
        with torch.device(DEV):
            layer = QATLinearComplexPhase(case["method"], case["method"], case["bits"] > 0, max(2, case["bits"]),
                                          case["rotate"], in_features=case["inf"], out_features=case["outf"])
        layer.weight.data, layer.bias.data = p["weight"], p["bias"]
        if case["rotate"]:
            layer.quantizer_u.rotation_angle.data.fill_(p["angles"][0])
            layer.quantizer_w.rotation_angle.data.fill_(p["angles"][1])
        layer.train()
        return {"kind": kind, "f": layer, "x": p["x"].requires_grad_(True), "gy": p["gy"], "amp": case["amp"]}
    return {"kind": kind, "conj": case["conj"], "block": case["block"], **_plane_params(g, case)}


def run(state):
    kind = state["kind"]
    if kind in ("model", "block", "layer"):
        with torch.no_grad():
            return state["f"](state["x"])
    if kind == "frozen":
        y = state["f"](state["x"])
        (gx,) = torch.autograd.grad(y, state["x"], state["gy"])
        return {"y": y.detach(), "gx": gx}
    if kind == "train":
        layer, x = state["f"], state["x"]
        x.grad = None
        layer.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.float16, enabled=state["amp"]):
            y = layer(x)
        y.backward(state["gy"])
        return {"y": y.detach(), "gx": x.grad, **{n: q.grad for n, q in layer.named_parameters()}}
    from quant_models import ops

    return ops.phase_linear(state["xr"], state["xi"], state["codes"], *state["gamma"], block=state["block"],
                            conj_x=state["conj"])


# ---------------------------------------------------------------------------
# the work, and how far a correct implementation may be off
# ---------------------------------------------------------------------------
def _layer_work(rows, inf, outf, size, book="axis2"):
    per, bits = BOOKS[book]
    codes = 2 * per * bits * (inf // 2) * (outf // 2) // 8
    return {"bytes": rows * (inf + outf) * size + codes + 40 * (outf // 2), "flops": 2 * rows * inf * outf}


def _add(*works):
    return {k: sum(w[k] for w in works) for k in ("bytes", "flops")}


def _block_work(images, tokens, dim, size, book):
    """A block reads its input once, writes its output once and reads its codes."""
    m = images * tokens
    w = _add(*(_layer_work(0, i, o, size, book) for i, o in
               ((dim, 3 * dim), (dim, dim), (dim, 4 * dim), (4 * dim, dim))))
    return {"bytes": w["bytes"] + 2 * m * dim * size, "flops": 24 * m * dim * dim + 4 * m * tokens * dim}


def work(case):
    kind = case["kind"]
    if kind == "model":
        tokens = (case["img"] // 16) ** 2 + (2 if case["model"] == "deit" else 1)
        block = _block_work(case["batch"], tokens, case["dim"], 2, case["book"])
        patches = case["batch"] * (case["img"] // 16) ** 2
        codes = _block_work(0, tokens, case["dim"], 2, case["book"])["bytes"]
        return {"bytes": case["depth"] * codes + 2 * case["batch"] * (3 * case["img"] ** 2 + 1000),
                "flops": case["depth"] * block["flops"] + 2 * patches * 768 * case["dim"]}
    size = 4 if kind in ("train", "plane") else 4 if case["dtype"] == "fp32" else 2
    if kind == "block":
        return _block_work(case["batch"], case["tokens"], case["dim"], size, case["book"])
    if kind == "plane":
        m, k, n = case["rows"], case["inf"], case["outf"]
        nblk = 1 if case["block"] == 0 else -(-k // case["block"])
        return {"bytes": 8 * m * k + n * k // 4 + 4 * n * nblk + 8 * m * n, "flops": 8 * m * k * n}
    rows, inf, outf = case["rows"], case["inf"], case["outf"]
    if kind == "layer":
        return _layer_work(rows, inf, outf, size, case["book"])
    if kind == "frozen":
        w = _layer_work(rows, inf, outf, size, case["book"])
        return {"bytes": 2 * w["bytes"], "flops": 2 * w["flops"]}
    # training: x, the output's gradient and the weight in; y and three gradients out
    out = 2 if case["amp"] else 4
    return {"bytes": 2 * rows * (4 * inf + out * outf) + 8 * inf * outf, "flops": 6 * rows * inf * outf}


def tolerance(case):
    kind = case["kind"]
    if kind == "plane":
        return {"rel": 2e-6, "max": 4e-5}
    if kind == "train" and not case["amp"]:
        # float32 sums; the rotation's gradient is one sum over the whole weight, with cancellation
        return {"rel": 1e-3, "max": 1e-2} if case["rotate"] else {"rel": 1e-5, "max": 1e-3}
    half = case.get("dtype") != "bf16"
    if kind == "model":
        return {"rel": 0.006, "max": 0.1}
    if kind == "block":
        # with quantized activations a rounding that tips a level moves a whole step
        return {"rel": 0.018 if case["bits"] else 0.002 if half else 0.0125, "max": 0.5 if case["bits"] else 0.1}
    if kind == "train":
        return {"rel": 1.5e-3, "max": 0.05}
    return {"rel": 1.5e-3 if half else 7e-3, "max": 0.05}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _unpack(plane, bits):
    parts = [(plane >> s) & ((1 << bits) - 1) for s in range(0, 8, bits)]
    return torch.stack(parts, dim=-1).reshape(plane.shape[0], -1).long()


def _plane_values(codes, s_re, s_im, book):
    s_re, s_im = s_re.double(), s_im.double()
    if book == "table":
        return torch.gather(s_re, 1, codes), torch.gather(s_im, 1, codes)
    if book == "psk16":
        a = codes.double() * (2 * math.pi / 16)
        return s_re * torch.cos(a), s_re * torch.sin(a)
    sign = torch.where(codes & 1 == 1, 1.0, -1.0).double()
    if book == "sign2":
        return s_re * sign, s_im * torch.where(codes & 2 == 2, 1.0, -1.0).double()
    on_im = codes & 2 == 2
    return torch.where(on_im, 0.0, s_re * sign), torch.where(on_im, s_im * sign, 0.0)


def _matrix(p):
    """The real [out, in] matrix of U x + W conj(x) on [re | im] features."""
    per, bits = BOOKS[p["book"]]
    uw = []
    for half in range(2):
        re = im = 0.0
        for plane, (s_re, s_im) in list(zip(p["planes"], p["scales"]))[half * per:(half + 1) * per]:
            v = _plane_values(_unpack(plane, bits), s_re, s_im, p["book"])
            re, im = re + v[0], im + v[1]
        if p["rotation"] is not None:
            c, s = p["rotation"][half]
            re, im = re * c - im * s, im * c + re * s
        uw.append((re, im))
    (ur, ui), (wr, wi) = uw
    return torch.cat((torch.cat((wr + ur, wi - ui), 1), torch.cat((wi + ui, ur - wr), 1)), 0)


def _fake_quant(x, bits):
    """Each half of a row on 2^bits levels of its largest magnitude."""
    if not bits:
        return x
    qmax, halves = float((1 << (bits - 1)) - 1), []
    for h in x.chunk(2, dim=-1):
        scale = qmax / h.abs().amax(dim=-1, keepdim=True).clamp_min(1e-5)
        halves.append((h * scale).round().clamp(-qmax - 1, qmax) / scale)
    return torch.cat(halves, dim=-1)


def _exact_linear(x, p, bits=0):
    return _fake_quant(x, bits) @ _matrix(p).t() + p["bias"].double()


def _exact_norm(x, wb):
    return F.layer_norm(x, x.shape[-1:], wb[0].double(), wb[1].double(), 1e-5)


def _exact_block(x, p, heads, bits):
    b, n, c = x.shape
    qkv = _exact_linear(_exact_norm(x, p["norm1"]), p["qkv"], bits)
    q, k, v = (t.contiguous() for t in qkv.reshape(b, n, 3, heads, c // heads).permute(2, 0, 3, 1, 4).unbind(0))
    mixed = []
    for lo in range(0, b, 32):  # the score matrices of 32 images at a time
        s = q[lo:lo + 32] @ k[lo:lo + 32].transpose(-1, -2).contiguous() / math.sqrt(c // heads)
        mixed.append(torch.softmax(s, dim=-1) @ v[lo:lo + 32])
    x = x + _exact_linear(torch.cat(mixed).transpose(1, 2).reshape(b, n, c), p["proj"], bits)
    h = F.gelu(_exact_linear(_exact_norm(x, p["norm2"]), p["fc1"], bits))
    return x + _exact_linear(h, p["fc2"], bits)


def _exact_model(case, p):
    x, dim = p["x"].double(), case["dim"]
    b, side = x.shape[0], case["img"] // 16
    patches = x.reshape(b, 3, side, 16, side, 16).permute(0, 2, 4, 1, 3, 5).reshape(b, side * side, 768)
    x = patches @ p["patch"][0].double().reshape(dim, -1).t() + p["patch"][1].double()
    x = torch.cat([t.double().expand(b, 1, dim) for t in p["prefix"]] + [x], dim=1) + p["pos"].double()
    for block in p["blocks"]:
        x = _exact_block(x, block, case["heads"], 0)
    x = _exact_norm(x, p["norm"])
    return sum(_exact_linear(x[:, i], head) for i, head in enumerate(p["heads"])) / len(p["heads"])


def _stage(re, im, kind):
    """One float32 stage of the training quantizer: the layer's codes are
    decided in float32, its scales are means over the whole plane."""
    def mean(v, mask, floor):
        return (v.abs().double() * mask).sum().div(mask.sum().clamp_min(1)).float().clamp_min(floor)

    if kind == "sign":
        ones = torch.ones_like(re)
        return (torch.where(re >= 0, 1.0, -1.0) * mean(re, ones, 1e-6),
                torch.where(im >= 0, 1.0, -1.0) * mean(im, ones, 1e-6))
    on_re = re.abs() > im.abs()
    on_im = im.abs() > re.abs()
    tie = ~(on_re | on_im)
    on_re = on_re | (tie & ((re * im < 0) | ((re == 0) & (im == 0))))
    sr, si = mean(re, on_re, 1e-5), mean(im, ~on_re, 1e-5)
    return (torch.where(on_re, torch.where(re >= 0, 1.0, -1.0) * sr, 0.0),
            torch.where(on_re, 0.0, torch.where(im >= 0, 1.0, -1.0) * si))


def _exact_train(case, p):
    w = p["weight"]
    no, ni = w.shape[0] // 2, w.shape[1] // 2
    a11, a12, a21, a22 = w[:no, :ni], w[:no, ni:], w[no:, :ni], w[no:, ni:]
    planes = [(0.5 * (a11 + a22), 0.5 * (a21 - a12)), (0.5 * (a11 - a22), 0.5 * (a12 + a21))]
    kind = "sign" if "new" in case["method"] else "axis"
    steps = {"complex_phase_v1": 1, "complex_phase_v2": 2, "complex_phase_new_v2": 2, "complex_phase_v4": 4}[case["method"]]
    quantized = []
    for i, (re, im) in enumerate(planes):
        if case["rotate"]:
            t = torch.tensor(p["angles"][i], device=DEV)
            c, s = torch.cos(t), torch.sin(t)
            re, im = re * c + im * s, im * c - re * s
        q_re, q_im = torch.zeros_like(re), torch.zeros_like(im)
        for _ in range(steps):
            s_re, s_im = _stage(re, im, kind)
            q_re, q_im, re, im = q_re + s_re, q_im + s_im, re - s_re, im - s_im
        if case["rotate"]:
            q_re, q_im = q_re * c - q_im * s, q_im * c + q_re * s
        quantized.append((q_re.double(), q_im.double()))
    (ur, ui), (wr, wi) = quantized
    a = torch.cat((torch.cat((wr + ur, wi - ui), 1), torch.cat((wi + ui, ur - wr), 1)), 0)
    x, gy = _fake_quant(p["x"], case["bits"]).double(), p["gy"].double()
    out = {"y": x @ a.t() + p["bias"].double(), "gx": gy @ a, "weight": gy.t().contiguous() @ x, "bias": gy.sum(0)}
    if case["rotate"]:
        g = out["weight"]
        g11, g12, g21, g22 = g[:no, :ni], g[:no, ni:], g[no:, :ni], g[no:, ni:]
        grads = ((g11 + g22, g21 - g12), (g11 - g22, g12 + g21))
        for name, (g_re, g_im), (re, im), (q_re, q_im) in zip("uw", grads, planes, quantized):
            th = (g_re * (im.double() - q_im) + g_im * (q_re - re.double())).sum()
            out["quantizer_%s.rotation_angle" % name] = th.reshape(1)
    return out


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    with torch.no_grad():
        if kind == "model":
            return _exact_model(case, _model_params(g, case))
        if kind == "block":
            dtype = DTYPES[case["dtype"]]
            p = _block_params(g, case["dim"], case["book"], case["rotate"], dtype)
            x = _normal(g, case["batch"], case["tokens"], case["dim"]).to(dtype)
            return _exact_block(x.double(), p, case["heads"], case["bits"])
        if kind in ("layer", "frozen"):
            dtype = DTYPES[case["dtype"]]
            p = _codes(g, case["outf"], case["inf"], case["book"], case["rotate"])
            x = _normal(g, case["rows"], case["inf"]).to(dtype)
            y = _exact_linear(_fake_quant(x.float(), case["bits"]).double(), p)
            if kind == "layer":
                return y
            gy = _normal(g, case["rows"], case["outf"], scale=0.1).to(dtype)
            return {"y": y, "gx": gy.double() @ _matrix(p)}
        if kind == "train":
            return _exact_train(case, _train_params(g, case))
        p, k = _plane_params(g, case), case["inf"]
        c = _unpack(p["codes"], 2)
        block = case["block"] or k
        sr, si = ((1.0 / t.double()).repeat_interleave(block, dim=1)[:, :k] for t in p["gamma"])
        wr, wi = _plane_values(c, sr, si, "axis2")
        xr, xi = p["xr"].double(), p["xi"].double()
        if not case["conj"]:
            xi = -xi
        return xr @ wr.t() + xi @ wi.t(), xr @ wi.t() - xi @ wr.t()
