"""The work that programs have this library do, as cases that can be timed and compared.

Every case goes through the public entry points: torch functions and modules on tensors of the "omarchy_mac_torch"
device, autograd for the backward, torch.compile(backend="omarchy_mac_torch") and the fused stacks. Kinds:

    conv    one 2-D convolution: forward alone (inference), or forward and backward (grad input, weight and bias)
    dw      one depthwise convolution, forward and backward
    bn      one training BatchNorm + ReLU, forward and backward
    pool    one max pool, forward and backward
    linear  one fully connected layer, forward and backward
    cnn     PlainCNN: batch inference in eval mode, or one training step (SGD with momentum), as a fused stack
    block   one inverted-residual block (expand, depthwise, squeeze-excite, project), a compiled training step
    resnet  ResNet-18, a compiled training step (SGD with momentum)

A training step returns its logits and the optimizer's momentum buffers, which after the first step are the gradients.
"""

import math
import pathlib
import sys

import torch
import torch.nn.functional as F

_PKG = str(pathlib.Path(__file__).resolve().parent.parent / "omarchy-mac-torch_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import omarchy_mac_torch as omt  # noqa: E402
from omarchy_mac_torch import models  # noqa: E402

DEV = omt.DEVICE


def _conv(name, n, ci, co, h, w, ks, stride, pad, train=True, bias=False, layout="nchw"):
    return {"name": name, "kind": "conv", "n": n, "ci": ci, "co": co, "h": h, "w": w, "ks": ks, "stride": stride,
            "pad": pad, "train": train, "bias": bias, "layout": layout}


def listed():
    return [
        # a ResNet body's 3x3 layer at the batch of large-scale training, the largest images and filters of its stages
        _conv("conv3x3_56_b256", 256, 64, 64, 56, 56, 3, 1, 1),
        # its 1x1 expansion: a short reduction, four times as many outputs as inputs
        _conv("conv1x1_28_b256", 256, 128, 512, 28, 28, 1, 1, 0),
        # the same body trained channels_last, a late stage
        _conv("conv3x3_14_b256_nhwc", 256, 256, 256, 14, 14, 3, 1, 1, layout="nhwc"),
        # a downsampling layer of a net with sizes of its own: ragged batch, channels and planes, a bias
        _conv("conv3x3_s2_ragged", 37, 120, 200, 45, 39, 3, 2, 1, bias=True),
        # AlexNet's first layer: 3 input channels, 11x11, stride 4
        _conv("conv11x11_stem_b16", 16, 3, 64, 224, 224, 11, 4, 2, bias=True),
        # a depthwise layer of a mobile net
        {"name": "dw5x5_28_b32", "kind": "dw", "n": 32, "c": 96, "h": 28, "w": 28, "ks": 5, "stride": 1},
        # normalization over a large early-stage activation
        {"name": "bn_relu_56_b256", "kind": "bn", "n": 256, "c": 64, "h": 56, "w": 56},
        # the pool after a 7x7 stem at full image size
        {"name": "maxpool3_112_b32", "kind": "pool", "n": 32, "c": 64, "h": 112, "w": 112, "ks": 3, "stride": 2, "pad": 1},
        # a classifier head
        {"name": "linear_512_1000", "kind": "linear", "n": 128, "inp": 512, "out": 1000},
        # serving one image: the smallest calls, where the host and the launches count
        {"name": "plaincnn_infer_b1", "kind": "cnn", "n": 1, "size": 32, "train": False},
        # a mobile net's squeeze-excite block in training
        {"name": "se_block_28_b32", "kind": "block", "n": 32, "c": 40, "exp": 240, "h": 28, "w": 28, "ks": 5},
        # a whole training step of a small-image classifier
        {"name": "resnet18_step_b32", "kind": "resnet", "n": 32, "size": 64},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _channels(rng, lo, hi):
    c = _log(rng, lo, hi)
    step = rng.choice([1, 8, 16, 32, 64])  # most nets use round widths; pruned ones any width
    return c if c < step else c // step * step


def draw(rng):
    kind = rng.choice(["conv"] * 6 + ["dw", "bn", "pool", "linear", "cnn", "cnn"])
    if kind == "conv":
        ks = rng.choice([1, 1, 3, 3, 3, 3, 5, 7])
        stride = rng.choice([1, 1, 1, 2])
        ci, co = _channels(rng, 3, 768), _channels(rng, 8, 768)
        h, w = _log(rng, 7, 112), _log(rng, 7, 112)
        if rng.random() < 0.5:
            w = h
        case = {"kind": "conv", "n": _log(rng, 1, 256), "ci": ci, "co": co, "h": h, "w": w, "ks": ks, "stride": stride,
                "pad": ks // 2, "train": rng.random() < 0.8, "bias": rng.random() < 0.3,
                "layout": "nhwc" if rng.random() < 0.25 else "nchw"}
        while work(case)["flops"] > 150e9 or work(case)["bytes"] > 1.5e9:
            case["n"] = max(1, case["n"] // 2)
            if case["n"] == 1:
                case["ci"], case["co"] = max(3, case["ci"] // 2), max(8, case["co"] // 2)
        return case
    h = _log(rng, 7, 112)
    w = h if rng.random() < 0.6 else _log(rng, 7, 112)
    if kind in ("dw", "bn", "pool"):
        c, n = _channels(rng, 8, 512), _log(rng, 1, 256)
        case = {"kind": kind, "n": n, "c": c, "h": h, "w": w}
        if kind == "dw":
            case.update(ks=rng.choice([3, 5, 7]), stride=rng.choice([1, 1, 1, 2]))
        if kind == "pool":
            case.update(zip(("ks", "stride", "pad"), rng.choice([(2, 2, 0), (3, 2, 1)])))
        while work(case)["bytes"] > 1.2e9:
            case["n"] = max(1, case["n"] // 2)
        return case
    if kind == "linear":
        return {"kind": kind, "n": _log(rng, 1, 1024), "inp": _channels(rng, 64, 4096), "out": _channels(rng, 10, 4096)}
    return {"kind": "cnn", "n": _log(rng, 1, 256), "size": rng.choice([28, 32, 48, 64]), "train": rng.random() < 0.5}


# ---- inputs ---------------------------------------------------------------------------------------------------------

def _out(h, ks, s, p):
    return (h + 2 * p - ks) // s + 1


def _layer_inputs(case, seed):
    """Seeded tensors of a single layer: activations as a ReLU leaves them (an image's for 3 channels), Kaiming
    weights, a gradient of the size a mean loss over the batch hands back."""
    torch.manual_seed(seed)
    kind, n = case["kind"], case["n"]

    def randn(*shape):
        return torch.randn(shape, device=DEV)

    if kind == "linear":
        return {"x": randn(n, case["inp"]).relu_(), "w": randn(case["out"], case["inp"]) * case["inp"] ** -0.5,
                "b": randn(case["out"]) * 0.1, "g": randn(n, case["out"]) / n}
    h, w = case["h"], case["w"]
    if kind == "conv":
        ci, co, ks, s, p = (case[k] for k in ("ci", "co", "ks", "stride", "pad"))
        x = randn(n, ci, h, w)
        x = x if ci == 3 else x.relu_()
        t = {"x": x, "w": randn(co, ci, ks, ks) * (2.0 / (ci * ks * ks)) ** 0.5}
        if case["bias"]:
            t["b"] = randn(co) * 0.1
        if case["train"]:
            t["g"] = randn(n, co, _out(h, ks, s, p), _out(w, ks, s, p)) / n
        if case["layout"] == "nhwc":
            t = {k: v.contiguous(memory_format=torch.channels_last) if v.dim() == 4 else v for k, v in t.items()}
        return t
    c = case["c"]
    if kind == "dw":
        ks, s = case["ks"], case["stride"]
        return {"x": randn(n, c, h, w).relu_(), "w": randn(c, 1, ks, ks) * (2.0 / (ks * ks)) ** 0.5,
                "g": randn(n, c, _out(h, ks, s, ks // 2), _out(w, ks, s, ks // 2)) / n}
    if kind == "bn":
        return {"x": randn(n, c, h, w) * 0.7 + 0.2, "w": randn(c) * 0.1 + 1.0, "b": randn(c) * 0.1,
                "g": randn(n, c, h, w) / n}
    ks, s, p = case["ks"], case["stride"], case["pad"]
    return {"x": randn(n, c, h, w).relu_(), "g": randn(n, c, _out(h, ks, s, p), _out(w, ks, s, p)) / n}


def _model_inputs(case, seed):
    """Host tensors: a batch of images (a block: its input activation) and labels."""
    g = torch.Generator().manual_seed(seed)
    if case["kind"] == "block":
        shape = (case["n"], case["c"], case["h"], case["w"])
        return torch.randn(shape, generator=g), torch.randn(shape, generator=g) / case["n"]
    classes = 1000 if case["kind"] == "resnet" else 10
    return (torch.randn((case["n"], 3, case["size"], case["size"]), generator=g),
            torch.randint(0, classes, (case["n"],), generator=g))


def _new_model(case):
    """The model on the host, its weights the same for every batch of the case; a served one has seen training data
    (running statistics, affine parameters)."""
    torch.manual_seed(7)
    if case["kind"] == "resnet":
        return models.resnet18(1000)
    if case["kind"] == "block":
        return models._kaiming(models.InvertedResidual(case["c"], case["exp"], case["c"], case["ks"], True))
    net = models.plain_cnn(10)
    if not case["train"]:
        for m in net.modules():
            if isinstance(m, torch.nn.BatchNorm2d):
                m.running_mean.normal_(0.0, 0.2)
                m.running_var.uniform_(0.5, 1.5)
                torch.nn.init.uniform_(m.weight, 0.8, 1.2)
                torch.nn.init.normal_(m.bias, 0.0, 0.1)
        net.eval()
    return net


# A program has one model that it feeds many batches: one per case and process. prepare() sets it back to its first
# weights.
_MODELS = {}


def _device_model(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _MODELS:
        base = _new_model(case)
        start = {k: v.clone() for k, v in base.state_dict().items()}
        model = base.to(DEV)
        call = model
        if case["kind"] in ("block", "resnet"):
            call = torch.compile(model, backend=DEV, dynamic=False)
        opt = torch.optim.SGD(model.parameters(), lr=0.01, momentum=0.9)
        _MODELS[key] = (model, call, opt, start)
    model, call, opt, start = _MODELS[key]
    model.load_state_dict(start)
    for p in model.parameters():
        p.grad = None
        buf = opt.state.get(p, {}).get("momentum_buffer")
        if buf is not None:
            buf.zero_()
    return model, call, opt


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("cnn", "block", "resnet"):
        model, call, opt = _device_model(case)
        x, t = _model_inputs(case, seed)
        return {"case": case, "model": model, "call": call, "opt": opt, "x": x.to(DEV), "t": t.to(DEV)}
    s = {"case": case, **_layer_inputs(case, seed)}
    if kind == "bn":
        s["rm"], s["rv"] = torch.zeros(case["c"], device=DEV), torch.ones(case["c"], device=DEV)
    if kind != "conv" or case["train"]:
        for k in ("x", "w", "b"):
            if k in s:
                s[k].requires_grad_(True)
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "conv" and not case["train"]:
        with torch.no_grad():
            return {"y": F.conv2d(s["x"], s["w"], s.get("b"), case["stride"], case["pad"])}
    if kind == "cnn" and not case["train"]:
        with torch.no_grad():
            return {"logits": s["call"](s["x"])}
    if kind in ("cnn", "resnet"):
        logits = s["call"](s["x"])
        F.cross_entropy(logits, s["t"]).backward()
    elif kind == "block":
        logits = s["call"](s["x"])
        logits.backward(s["t"])
    if kind in ("cnn", "resnet", "block"):
        opt = s["opt"]
        opt.step()
        opt.zero_grad(set_to_none=True)
        return {"logits": logits.detach(),
                "momentum": [opt.state[p]["momentum_buffer"] for p in s["model"].parameters()]}
    if kind == "bn":
        y = F.relu(F.batch_norm(s["x"], s["rm"], s["rv"], s["w"], s["b"], True, 0.1, 1e-5))
    elif kind == "conv":
        y = F.conv2d(s["x"], s["w"], s.get("b"), case["stride"], case["pad"])
    elif kind == "dw":
        y = F.conv2d(s["x"], s["w"], None, case["stride"], case["ks"] // 2, 1, case["c"])
    elif kind == "linear":
        y = F.linear(s["x"], s["w"], s["b"])
    else:
        y = F.max_pool2d(s["x"], case["ks"], case["stride"], case["pad"])
    names = [k for k in ("x", "w", "b") if k in s]
    out = {"y": y.detach()}
    out.update(zip(("g" + k for k in names), torch.autograd.grad(y, [s[k] for k in names], s["g"])))
    if kind == "bn":
        out["rm"], out["rv"] = s["rm"], s["rv"]
    return out


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _conv_work(n, ci, co, h, w, ks, s, p, groups=1):
    oh, ow = _out(h, ks, s, p), _out(w, ks, s, p)
    x, wt, y = n * ci * h * w, co * (ci // groups) * ks * ks, n * co * oh * ow
    return x, wt, y, 2 * n * co * oh * ow * (ci // groups) * ks * ks


def _model_work(case):
    """Forward work of the model's convolutions and linear layers, from their shapes; activations and weights once."""
    flops = acts = weights = 0
    layers = []
    if case["kind"] == "block":
        n, c, e, h, w, ks = (case[k] for k in ("n", "c", "exp", "h", "w", "ks"))
        layers = [(n, c, e, h, w, 1, 1, 0, 1), (n, e, e, h, w, ks, 1, ks // 2, e), (n, e, c, h, w, 1, 1, 0, 1)]
    elif case["kind"] == "resnet":
        n, h = case["n"], _out(case["size"], 7, 2, 3)
        layers = [(n, 3, 64, case["size"], case["size"], 7, 2, 3, 1)]
        h, c = _out(h, 3, 2, 1), 64
        for wd, s in ((64, 1), (128, 2), (256, 2), (512, 2)):
            o = _out(h, 3, s, 1)
            layers += [(n, c, wd, h, h, 3, s, 1, 1)] + [(n, wd, wd, o, o, 3, 1, 1, 1)] * 3
            if s != 1:
                layers.append((n, c, wd, h, h, 1, s, 0, 1))
            h, c = o, wd
        layers.append((n, c, 1000, 1, 1, 1, 1, 0, 1))
    else:
        n, h, c = case["n"], case["size"], 3
        for wd in (32, 64, 128, 256):
            layers.append((n, c, wd, h, h, 3, 1, 1, 1))
            h, c = h // 2, wd
        layers.append((n, c, 10, 1, 1, 1, 1, 0, 1))
    for a in layers:
        x, wt, y, f = _conv_work(*a)
        flops, acts, weights = flops + f, acts + x + y, weights + wt
    return flops, acts, weights


def work(case):
    kind = case["kind"]
    if kind in ("cnn", "block", "resnet"):
        flops, acts, weights = _model_work(case)
        # training: every activation and its gradient written and read; a weight, its momentum and its gradient
        return ({"bytes": 4 * (2 * acts + 5 * weights), "flops": 3 * flops} if case.get("train", True)
                else {"bytes": 4 * (acts + weights), "flops": flops})
    if kind == "linear":
        n, i, o = case["n"], case["inp"], case["out"]
        return {"bytes": 4 * (2 * n * i + 2 * n * o + 2 * i * o + 2 * o), "flops": 6 * n * i * o}
    n, h, w = case["n"], case["h"], case["w"]
    if kind in ("conv", "dw"):
        if kind == "dw":
            x, wt, y, f = _conv_work(n, case["c"], case["c"], h, w, case["ks"], case["stride"], case["ks"] // 2,
                                     case["c"])
        else:
            x, wt, y, f = _conv_work(n, case["ci"], case["co"], h, w, case["ks"], case["stride"], case["pad"])
        if not case.get("train", True):
            return {"bytes": 4 * (x + wt + y), "flops": f}
        return {"bytes": 4 * (2 * x + 2 * wt + 2 * y), "flops": 3 * f}  # y, gx, gw written; x, w, gy read
    x = n * case["c"] * h * w
    if kind == "bn":
        return {"bytes": 4 * 4 * x, "flops": 15 * x}  # x and gy read, y and gx written
    y = n * case["c"] * _out(h, case["ks"], case["stride"], case["pad"]) * _out(w, case["ks"], case["stride"],
                                                                               case["pad"])
    return {"bytes": 4 * (2 * x + 2 * y), "flops": y * case["ks"] ** 2}


# ---- how far another correct implementation may be off --------------------------------------------------------------

def tolerance(case):
    kind = case["kind"]
    if kind == "pool":
        return {"rel": 1e-7}  # selected values; a gradient adds at most four terms
    if kind == "resnet" or (kind == "cnn" and case["train"]):
        # rounding moves a few activations across a ReLU or to another of a pool's taps; each moves the gradients of
        # all layers before it: up to 3.6e-3 from the 64-bit gradients as measured
        return {"rel": 1e-2, "max": 0.9}
    if kind == "block":
        return {"rel": 1e-3, "max": 0.9}  # the same in the squeeze-excite's hidden layer: up to 6e-5 as measured
    if kind == "bn":
        return {"rel": 2e-6, "max": 0.9}  # the largest difference is a ReLU mask at a zero crossing
    # 32-bit sums of up to millions of terms (weight gradients) in any order: up to 1e-6 from the 64-bit ones
    return {"rel": 1e-5, "max": 1e-3}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------

def _host64(t):
    return t.detach().cpu().double()


def _dev64(t):
    return t.detach().cpu().cuda().double()


def _exact_conv(case, t):
    """Tap by tap: y += W_tap x_tap; gx_tap += W_tap' gy; gw_tap = gy x_tap'."""
    x, w = _dev64(t["x"]).contiguous(), _dev64(t["w"]).contiguous()
    n, ci, h, wd = x.shape
    co, ks, s, p = w.shape[0], case["ks"], case["stride"], case["pad"]
    oh, ow = _out(h, ks, s, p), _out(wd, ks, s, p)
    train = case["train"]
    g = _dev64(t["g"]).contiguous().reshape(n, co, oh * ow) if train else None
    y = torch.zeros((n, co, oh * ow), dtype=torch.float64, device=x.device)
    gw = torch.zeros_like(w) if train else None
    gx = torch.zeros((n, ci, h + 2 * p, wd + 2 * p), dtype=torch.float64, device=x.device) if train else None
    xp = F.pad(x, (p, p, p, p))
    del x
    step = max(1, (1 << 28) // max(1, max(ci, co) * oh * ow))  # images at a time: at most 2 GB of 64-bit values
    for n0 in range(0, n, step):
        for ky in range(ks):
            for kx in range(ks):
                at = (slice(n0, n0 + step), slice(None), slice(ky, ky + s * (oh - 1) + 1, s),
                      slice(kx, kx + s * (ow - 1) + 1, s))
                xs = xp[at].reshape(-1, ci, oh * ow)
                wt = w[:, :, ky, kx].contiguous()
                y[n0:n0 + step] += torch.matmul(wt, xs)
                if train:
                    gs = g[n0:n0 + step]
                    gx[at] += torch.matmul(wt.t().contiguous(), gs).reshape(-1, ci, oh, ow)
                    gw[:, :, ky, kx] += gs.transpose(0, 1).reshape(co, -1) @ xs.permute(0, 2, 1).reshape(-1, ci)
    if "b" in t:
        y += _dev64(t["b"])[:, None]
    out = {"y": y.reshape(n, co, oh, ow)}
    if train:
        out.update(gx=gx[:, :, p:p + h, p:p + wd], gw=gw)
        if "b" in t:
            out["gb"] = g.sum((0, 2))
    return out


def _exact_dw(case, t):
    x, w, g = _dev64(t["x"]), _dev64(t["w"]), _dev64(t["g"])
    n, c, h, wd = x.shape
    ks, s = case["ks"], case["stride"]
    p = ks // 2
    oh, ow = g.shape[2:]
    xp = F.pad(x, (p, p, p, p))
    y, gxp, gw = torch.zeros_like(g), torch.zeros_like(xp), torch.zeros_like(w)
    for ky in range(ks):
        for kx in range(ks):
            at = (slice(None), slice(None), slice(ky, ky + s * (oh - 1) + 1, s), slice(kx, kx + s * (ow - 1) + 1, s))
            tap = w[:, 0, ky, kx][:, None, None]
            y += xp[at] * tap
            gxp[at] += g * tap
            gw[:, 0, ky, kx] = (xp[at] * g).sum((0, 2, 3))
    return {"y": y, "gx": gxp[:, :, p:p + h, p:p + wd], "gw": gw}


def _exact_bn(t):
    x, w, b, g = (_dev64(t[k]) for k in ("x", "w", "b", "g"))
    m = x.numel() // x.shape[1]
    mean = x.mean((0, 2, 3))
    var = (x - mean[:, None, None]).square().mean((0, 2, 3))
    xh = (x - mean[:, None, None]) * (var + 1e-5).rsqrt()[:, None, None]
    y = (xh * w[:, None, None] + b[:, None, None]).clamp_min(0)
    g = g * (y > 0)
    gb, gw = g.sum((0, 2, 3)), (g * xh).sum((0, 2, 3))
    gx = (w * (var + 1e-5).rsqrt())[:, None, None] * (g - gb[:, None, None] / m - xh * (gw[:, None, None] / m))
    return {"y": y, "gx": gx, "gw": gw, "gb": gb, "rm": 0.1 * mean, "rv": 0.9 + 0.1 * var * m / (m - 1)}


def _exact_pool(case, t):
    x, g = _dev64(t["x"]), _dev64(t["g"])
    y, at = F.max_pool2d(x, case["ks"], case["stride"], case["pad"], return_indices=True)
    gx = torch.zeros_like(x).flatten(2).scatter_add_(2, at.flatten(2), g.flatten(2)).reshape(x.shape)
    return {"y": y, "gx": gx}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("cnn", "block", "resnet"):
        if kind == "cnn" and case["n"] * case["size"] ** 2 > 256 * 1024:
            return None  # a minute and more on the host
        model = _new_model(case).double()
        x, t = _model_inputs(case, seed)
        logits = model(x.double())
        if not case.get("train", True):
            return {"logits": logits.detach()}
        if kind == "block":
            logits.backward(t.double())
        else:
            F.cross_entropy(logits, t).backward()
        return {"logits": logits.detach(), "momentum": [p.grad for p in model.parameters()]}
    t = _layer_inputs(case, seed)
    if kind == "conv":
        return _exact_conv(case, t)
    if kind == "dw":
        return _exact_dw(case, t)
    if kind == "bn":
        return _exact_bn(t)
    if kind == "pool":
        return _exact_pool(case, t)
    x, w, b, g = (_host64(t[k]) for k in ("x", "w", "b", "g"))
    return {"y": x @ w.t() + b, "gx": g @ w, "gw": g.t() @ x, "gb": g.sum(0)}
