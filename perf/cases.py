"""The work a program has this backend do, as cases that can be timed.

Every case runs FP32 torch operators on "vulkan" tensors, the way a training
or inference program on this backend does: single layers and blocks forward
and backward, the optimizer step, and one whole network forward.  ``listed()``
names twelve of them, ``draw()`` gives others from the same ranges, and
``exact()`` restates a case in float64 with stock torch.

Case fields: ``kind`` selects the path, the others are its sizes.
"""
from __future__ import annotations

import math
import os
import sys

import torch
from torch import nn
from torch.nn import functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pytorch-vulkan_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)


def listed():
    return [
        # Classifier head while serving a handful of requests: 8 rows, so the
        # weight is read once for almost no arithmetic and latency counts.
        dict(name="linear_head_infer", kind="linear", m=8, k=2048, n=1000, train=False),
        # One training step of the largest dense layer (8192 rows, 4096 x 4096).
        dict(name="linear_train", kind="linear", m=8192, k=4096, n=4096, train=True),
        # 3x3 layer of a residual network, forward and all gradients, small batch.
        dict(name="conv3x3_train", kind="conv", n=8, cin=64, cout=64, h=56, w=56, k=3, s=1, groups=1, train=True,
             dx=True),
        # 1x1 expansion of a bottleneck block at batch 64.
        dict(name="conv1x1_train", kind="conv", n=64, cin=128, cout=512, h=28, w=28, k=1, s=1, groups=1, train=True,
             dx=True),
        # First layer of an image network: three channels, 7x7, stride 2; no input gradient.
        dict(name="conv7x7_stem_train", kind="conv", n=64, cin=3, cout=64, h=224, w=224, k=7, s=2, groups=1,
             train=True, dx=False),
        # Down-sampling layer between two U-Net levels.
        dict(name="conv3x3_s2_train", kind="conv", n=16, cin=256, cout=256, h=32, w=32, k=3, s=2, groups=1,
             train=True, dx=True),
        # Depthwise layer (one filter per channel), forward and all gradients.
        dict(name="conv_depthwise_train", kind="conv", n=32, cin=192, cout=192, h=28, w=28, k=3, s=1, groups=192,
             train=True, dx=True),
        # Self-attention over a 16x16 feature map: 4 heads of 64, batch 16.
        dict(name="attention_train", kind="attention", b=16, heads=4, tokens=256, dim=64),
        # Batch normalisation and ReLU behind a bottleneck's reduction layer.
        dict(name="batchnorm_relu_train", kind="batchnorm", n=64, c=128, h=28, w=28),
        # Optimizer step over a residual network's parameters (25.6 M in 161
        # tensors, a third of them vectors), parameters and moments as views
        # of flat buffers.
        dict(name="adamw_step", kind="adamw", total=25557032, tensors=161, align=64, amsgrad=False),
        # Residual block of the U-Net (GroupNorm, SiLU, 3x3, twice), training.
        dict(name="resblock_train", kind="resblock", n=16, cin=256, cout=256, h=32, w=32),
        # One denoising call of a sampler: the whole U-Net on a single image.
        dict(name="unet_infer", kind="unet", n=1, base=128, image=64),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "conv", "conv", "conv", "conv", "depthwise", "attention", "groupnorm",
                       "batchnorm", "adamw", "resblock", "unet"])
    if kind == "linear":
        return dict(kind=kind, m=_log(rng, 1, 8192), k=_log(rng, 64, 4096), n=_log(rng, 64, 4096),
                    train=rng.random() < 0.7)
    if kind == "conv":
        groups = rng.choice([1, 1, 1, 1, 2, 4, 8])
        cin = _log(rng, 3, 1024) if groups == 1 else groups * _log(rng, 4, 64)
        cout = _log(rng, 16, 1024) if groups == 1 else groups * _log(rng, 4, 64)
        k, s = rng.choice([1, 1, 3, 3, 3, 5, 7]), rng.choice([1, 1, 2])
        h = _log(rng, 7, 112)
        w = h if rng.random() < 0.5 else _log(rng, 7, 112)
        n = _log(rng, 1, 64)
        train = rng.random() < 0.75
        while n > 1 and (2.0 * n * cout * (cin // groups) * k * k * h * w / (s * s) > 3e10
                         or n * max(cin, cout) * h * w > 3e7):
            n //= 2
        while h * w * max(cin, cout) > 3e7 or 2.0 * cout * (cin // groups) * k * k * h * w / (s * s) > 3e10:
            h, w = max(7, h // 2), max(7, w // 2)
        return dict(kind=kind, n=n, cin=cin, cout=cout, h=h, w=w, k=k, s=s, groups=groups, train=train, dx=train)
    if kind == "depthwise":
        c, k, h = _log(rng, 16, 768), rng.choice([3, 3, 5]), _log(rng, 7, 56)
        n = min(_log(rng, 1, 64), max(1, int(2e7 / (c * h * h))))
        train = rng.random() < 0.6
        return dict(kind="conv", n=n, cin=c, cout=c, h=h, w=h, k=k, s=rng.choice([1, 1, 2]), groups=c, train=train,
                    dx=train)
    if kind == "attention":
        return dict(kind=kind, b=_log(rng, 1, 16), heads=rng.choice([1, 2, 4, 8]), tokens=_log(rng, 49, 576),
                    dim=rng.choice([32, 40, 64, 80, 128]))
    if kind == "groupnorm":
        g = rng.choice([8, 16, 32])
        h = _log(rng, 8, 64)
        return dict(kind=kind, n=_log(rng, 1, 16), c=g * _log(rng, 1, 16), groups=g, h=h, w=h)
    if kind == "batchnorm":
        c, h = _log(rng, 16, 2048), _log(rng, 7, 56)
        return dict(kind=kind, n=min(_log(rng, 2, 64), max(2, int(2e7 / (c * h * h)))), c=c, h=h, w=h)
    if kind == "adamw":
        total = _log(rng, 100000, 60000000)
        return dict(kind=kind, total=total, tensors=_log(rng, 4, 250), align=rng.choice([64, 64, 1]),
                    amsgrad=rng.random() < 0.3)
    if kind == "resblock":
        h = rng.choice([8, 12, 16, 24, 32, 48, 64])
        top = 512 if h <= 16 else 256 if h <= 32 else 128
        return dict(kind=kind, n=_log(rng, 1, 16), cin=32 * _log(rng, 1, top // 32), cout=32 * _log(rng, 2, top // 32),
                    h=h, w=h)
    return dict(kind=kind, n=_log(rng, 1, 4), base=32 * rng.randint(1, 4), image=rng.choice([32, 40, 48, 64]))


# ------------------------------------------------------------------ inputs
class _Gen:
    """float32 tensors made on the GPU from the seed alone, in call order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, scale=1.0, mean=0.0):
        return torch.randn(*shape, device="cuda", generator=self.g) * scale + mean

    def uniform(self, *shape, bound):
        return (torch.rand(*shape, device="cuda", generator=self.g) * 2 - 1) * bound

    def layer(self, *shape):
        """Weight and bias with the bounds torch.nn gives its layers."""
        bound = 1.0 / math.sqrt(math.prod(shape[1:]))
        return self.uniform(*shape, bound=bound), self.uniform(shape[0], bound=bound)


def _inputs(case, seed):
    """Named float32 CUDA tensors of one case (None where it has none)."""
    g, c = _Gen(seed), case
    kind = c["kind"]
    if kind == "linear":
        w, b = g.layer(c["n"], c["k"])
        return dict(x=g.normal(c["m"], c["k"]), w=w, b=b,
                    dy=g.normal(c["m"], c["n"], scale=0.05) if c["train"] else None)
    if kind == "conv":
        w, b = g.layer(c["cout"], c["cin"] // c["groups"], c["k"], c["k"])
        oh, ow = _out(c["h"], c), _out(c["w"], c)
        return dict(x=g.normal(c["n"], c["cin"], c["h"], c["w"]), w=w, b=b,
                    dy=g.normal(c["n"], c["cout"], oh, ow, scale=0.05) if c["train"] else None)
    if kind == "attention":
        bh = c["b"] * c["heads"]
        q, k, v, dy = (g.normal(bh, c["dim"], c["tokens"]) for _ in range(4))
        return dict(q=q, k=k, v=v, dy=dy * 0.05)
    if kind in ("groupnorm", "batchnorm"):
        shape = (c["n"], c["c"], c["h"], c["w"])
        return dict(x=g.normal(*shape, mean=0.3), w=g.normal(c["c"], scale=0.2, mean=1.0),
                    b=g.normal(c["c"], scale=0.2), dy=g.normal(*shape, scale=0.05),
                    rm=g.normal(c["c"], scale=0.1), rv=g.uniform(c["c"], bound=0.5) + 1.0)
    if kind == "adamw":
        n = c["total"]
        v = g.normal(n, scale=0.01).square_()
        return dict(p=g.normal(n, scale=0.05), g=g.normal(n, scale=0.01), m=g.normal(n, scale=0.003), v=v,
                    vmax=v * 1.25 if c["amsgrad"] else None)
    if kind == "resblock":
        return dict(x=g.normal(c["n"], c["cin"], c["h"], c["w"]),
                    dy=g.normal(c["n"], c["cout"], c["h"], c["w"], scale=0.05))
    return dict(x=g.normal(c["n"], 3, c["image"], c["image"]))


def _out(size, c):
    return (size + 2 * (c["k"] // 2) - c["k"]) // c["s"] + 1


def _sizes(case):
    """Element counts of the optimizer's parameters: a third of them vectors,
    the others matrices of growing size, the last one taking the rest."""
    n, total = case["tensors"], case["total"]
    mats = max(1, n - n // 3)
    vectors = [64 * (1 + i % 8) for i in range(n - mats)]
    room = max(mats, total - sum(vectors))
    weights = [1.0 + 3.0 * i / mats for i in range(mats)]
    a = case["align"]  # elements: where each tensor starts in the flat buffers
    sizes = [max(1, int(room * w / sum(weights)) // a * a or 1) for w in weights]
    sizes = [s for pair in zip(sizes, vectors) for s in pair] + sizes[len(vectors):] + vectors[mats:]
    sizes[-1] += max(0, total - sum(sizes))
    return sizes


def _fill(module, gen, to=lambda t: t):
    """Gives every parameter of a module made on the meta device its values:
    torch's default bounds for convolutions, unit scale for norms."""
    for m in module.modules():
        if isinstance(m, nn.Conv2d):
            w, b = gen.layer(*m.weight.shape)
        elif isinstance(m, nn.GroupNorm):
            w, b = gen.normal(m.num_channels, scale=0.1, mean=1.0), gen.normal(m.num_channels, scale=0.1)
        else:
            continue
        m.weight, m.bias = nn.Parameter(to(w)), nn.Parameter(to(b))
    return module


class _ResBlock(nn.Module):
    def __init__(self, cin, cout, groups):
        super().__init__()
        self.norm1, self.conv1 = nn.GroupNorm(groups, cin), nn.Conv2d(cin, cout, 3, padding=1)
        self.norm2, self.conv2 = nn.GroupNorm(groups, cout), nn.Conv2d(cout, cout, 3, padding=1)
        self.skip = nn.Conv2d(cin, cout, 1) if cin != cout else None

    def forward(self, x):
        h = self.conv1(F.silu(self.norm1(x)))
        h = self.conv2(F.silu(self.norm2(h)))
        return h + (self.skip(x) if self.skip is not None else x)


def _attend(q, k, v):
    """Attention over the columns of [batch * heads, dim, tokens] operands."""
    scores = torch.bmm(q.transpose(1, 2), k) * (q.shape[1] ** -0.5)
    return torch.bmm(v, torch.softmax(scores, dim=-1).transpose(1, 2))


class _Attention(nn.Module):
    def __init__(self, c, groups, heads=4):
        super().__init__()
        self.heads, self.norm = heads, nn.GroupNorm(groups, c)
        self.qkv, self.proj = nn.Conv2d(c, 3 * c, 1), nn.Conv2d(c, c, 1)

    def forward(self, x):
        b, c, h, w = x.shape
        qkv = self.qkv(self.norm(x)).reshape(b, 3, self.heads, c // self.heads, h * w)
        q, k, v = (qkv[:, i].reshape(b * self.heads, c // self.heads, h * w) for i in range(3))
        return x + self.proj(_attend(q, k, v).reshape(b, c, h, w))


class _UNet(nn.Module):
    """Diffusion U-Net: four levels (1, 2, 2, 4 times the base width), two
    residual blocks each, attention on the third."""

    def __init__(self, base, groups=32):
        super().__init__()
        widths = [base, 2 * base, 2 * base, 4 * base]
        self.first = nn.Conv2d(3, base, 3, padding=1)
        self.down, self.shrink, self.up, self.grow = (nn.ModuleList() for _ in range(4))
        c = base
        for i, wd in enumerate(widths):
            level = [_ResBlock(c, wd, groups), _ResBlock(wd, wd, groups)]
            self.down.append(nn.Sequential(*level, *([_Attention(wd, groups)] if i == 2 else [])))
            if i < 3:
                self.shrink.append(nn.Conv2d(wd, wd, 3, stride=2, padding=1))
            c = wd
        self.mid = _ResBlock(c, c, groups)
        for i in (3, 2, 1, 0):
            wd = widths[i]
            level = [_ResBlock(c + wd, wd, groups), _ResBlock(wd, wd, groups)]
            self.up.append(nn.Sequential(*level, *([_Attention(wd, groups)] if i == 2 else [])))
            if i:
                self.grow.append(nn.Conv2d(wd, wd, 3, padding=1))
            c = wd
        self.norm, self.last = nn.GroupNorm(groups, c), nn.Conv2d(c, 3, 3, padding=1)

    def forward(self, x):
        h, skips = self.first(x), []
        for i, level in enumerate(self.down):
            h = level(h)
            skips.append(h)
            h = self.shrink[i](h) if i < 3 else h
        h = self.mid(h)
        for i, level in enumerate(self.up):
            h = level(torch.cat([h, skips[3 - i]], 1))
            h = self.grow[i](F.interpolate(h, scale_factor=2.0, mode="nearest")) if i < 3 else h
        return self.last(F.silu(self.norm(h)))


def _module(case, to=lambda t: t, seed=0):
    with torch.device("meta"):
        if case["kind"] == "resblock":
            m = _ResBlock(case["cin"], case["cout"], 32)
        else:
            m = _UNet(case["base"])
    return _fill(m, _Gen(seed + 77777), to)


def _vulkan(t):
    return None if t is None else t.cpu().to("vulkan")


def prepare(case, seed):
    import torch_vulkan  # noqa: F401  (registers the device)
    from torch_vulkan.optim import AdamW

    t = {k: _vulkan(v) for k, v in _inputs(case, seed).items()}
    t["case"], kind = case, case["kind"]
    if kind in ("linear", "conv") and case["train"]:
        for k in ("x", "w", "b") if case.get("dx", True) else ("w", "b"):
            t[k].requires_grad_()
    elif kind == "attention":
        for k in "qkv":
            t[k].requires_grad_()
    elif kind in ("groupnorm", "batchnorm"):
        for k in "xwb":
            t[k].requires_grad_()
    elif kind == "adamw":
        params, at = [], 0
        for s in _sizes(case):
            p = t["p"][at:at + s].requires_grad_()
            p.grad = t["g"][at:at + s]
            params.append(p)
            at += s
        opt = AdamW(params, lr=1e-3, weight_decay=1e-2, amsgrad=case["amsgrad"])
        at = 0
        for p in params:
            s = p.numel()
            opt.state[p] = dict(step=9, exp_avg=t["m"][at:at + s], exp_avg_sq=t["v"][at:at + s])
            if case["amsgrad"]:
                opt.state[p]["max_exp_avg_sq"] = t["vmax"][at:at + s]
            at += s
        t["opt"] = opt
    elif kind in ("resblock", "unet"):
        t["module"] = _module(case, _vulkan, seed)
        if kind == "resblock":
            t["x"].requires_grad_()
    return t


def _forward(case, t):
    """The layer's output from its tensors, wherever they live."""
    kind = case["kind"]
    if kind == "linear":
        return F.linear(t["x"], t["w"], t["b"])
    if kind == "conv":
        return F.conv2d(t["x"], t["w"], t["b"], case["s"], case["k"] // 2, 1, case["groups"])
    if kind == "attention":
        return _attend(t["q"], t["k"], t["v"])
    if kind == "groupnorm":
        return F.silu(F.group_norm(t["x"], case["groups"], t["w"], t["b"]))
    return F.relu(F.batch_norm(t["x"], t["rm"], t["rv"], t["w"], t["b"], training=True))


def _step(case, t):
    """Outputs of one pass: the result and, in training, every gradient."""
    kind = case["kind"]
    if kind == "unet":
        with torch.no_grad():
            return [t["module"](t["x"])]
    if kind == "resblock":
        wanted = [t["x"], *t["module"].parameters()]
        y = t["module"](t["x"])
    elif kind in ("linear", "conv") and not case["train"]:
        with torch.no_grad():
            return [_forward(case, t)]
    else:
        wanted = [t[k] for k in ("q", "k", "v", "x", "w", "b") if k in t and t[k].requires_grad]
        y = _forward(case, t)
    out = [y.detach(), *torch.autograd.grad(y, wanted, t["dy"])]
    return out + [t["rm"], t["rv"]] if kind == "batchnorm" else out


def run(state):
    case = state["case"]
    if case["kind"] != "adamw":
        return _step(case, state)
    state["opt"].step()
    return [state[k] for k in ("p", "m", "v", "vmax") if state[k] is not None]


# ------------------------------------------------------------ in 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind in ("conv", "resblock", "unet"):
        if work(case)["flops"] > 4e11:
            return None
        dev = "cpu"  # float64 convolutions
    else:
        dev = "cuda"
    t = {k: None if v is None else v.to(dev, torch.float64) for k, v in _inputs(case, seed).items()}
    if kind == "adamw":
        b1, b2, lr, step = 0.9, 0.999, 1e-3, 10
        p = t["p"] * (1 - lr * 1e-2)
        m = t["m"] * b1 + t["g"] * (1 - b1)
        v = t["v"] * b2 + t["g"] * t["g"] * (1 - b2)
        top = torch.maximum(t["vmax"], v) if case["amsgrad"] else v
        p = p - lr / (1 - b1 ** step) * m / ((top / (1 - b2 ** step)).sqrt() + 1e-8)
        return [p, m, v] + ([top] if case["amsgrad"] else [])
    if kind in ("linear", "conv") and not case["train"]:
        return [_forward(case, t)]
    if kind in ("resblock", "unet"):
        t["module"] = _module(case, lambda x: x.to(dev, torch.float64), seed)
    for k in ("q", "k", "v", "x", "w", "b"):
        if k in t and kind != "unet" and (k != "x" or case.get("dx", True)):
            t[k].requires_grad_()
    return _step(case, t)


# ------------------------------------------------- bytes and operations
def _conv_flops(n, cin, cout, oh, ow, k, groups=1):
    return 2.0 * n * cout * oh * ow * (cin // groups) * k * k


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        m, k, n = c["m"], c["k"], c["n"]
        once, flops = m * k + n * k + n + m * n, 2.0 * m * n * k
        # Training also reads dy and writes the three gradients.
        return dict(bytes=4.0 * (once + (m * n + m * k + n * k + n if c["train"] else 0)),
                    flops=flops * (3 if c["train"] else 1))
    if kind == "conv":
        oh, ow = _out(c["h"], c), _out(c["w"], c)
        x, y = c["n"] * c["cin"] * c["h"] * c["w"], c["n"] * c["cout"] * oh * ow
        w = c["cout"] * (c["cin"] // c["groups"]) * c["k"] ** 2 + c["cout"]
        flops = _conv_flops(c["n"], c["cin"], c["cout"], oh, ow, c["k"], c["groups"])
        if not c["train"]:
            return dict(bytes=4.0 * (x + w + y), flops=flops)
        return dict(bytes=4.0 * (x + w + y + y + w + (x if c["dx"] else 0)), flops=flops * (3 if c["dx"] else 2))
    if kind == "attention":
        bh, t, d = c["b"] * c["heads"], c["tokens"], c["dim"]
        return dict(bytes=4.0 * 8 * bh * t * d, flops=6 * 2.0 * bh * t * t * d)
    if kind in ("groupnorm", "batchnorm"):
        e = c["n"] * c["c"] * c["h"] * c["w"]
        # Forward reads x and writes y, backward reads x and dy and writes dx.
        return dict(bytes=4.0 * 5 * e, flops=20.0 * e)
    if kind == "adamw":
        return dict(bytes=(36.0 if c["amsgrad"] else 28.0) * c["total"], flops=14.0 * c["total"])
    if kind == "resblock":
        n, ci, co, hw = c["n"], c["cin"], c["cout"], c["h"] * c["w"]
        flops = _conv_flops(n, ci, co, c["h"], c["w"], 3) + _conv_flops(n, co, co, c["h"], c["w"], 3)
        weights = 9 * ci * co + 9 * co * co
        if ci != co:
            flops += _conv_flops(n, ci, co, c["h"], c["w"], 1)
            weights += ci * co
        return dict(bytes=4.0 * (2 * n * (ci + co) * hw + 2 * weights), flops=3 * flops)
    # U-Net: shapes of every convolution and attention product on the meta device.
    total = dict(bytes=4.0 * 2 * 3 * c["n"] * c["image"] ** 2, flops=0.0)
    with torch.device("meta"):
        net = _UNet(c["base"])

        def conv(mod, inp, out):
            total["flops"] += 2.0 * out.numel() * mod.weight[0].numel()

        def attn(mod, inp, out):
            n, ch, h, w = out.shape
            total["flops"] += 4.0 * n * ch * (h * w) ** 2

        for mod in net.modules():
            if isinstance(mod, nn.Conv2d):
                mod.register_forward_hook(conv)
                total["bytes"] += 4.0 * (mod.weight.numel() + mod.bias.numel())
            elif isinstance(mod, _Attention):
                mod.register_forward_hook(attn)
        with torch.no_grad():
            net(torch.empty(c["n"], 3, c["image"], c["image"]))
    return total


def tolerance(case):
    # Distance from float64 seen on this path: up to 1.6e-6 for sums of 8192
    # FP32 terms in sequence, 0.9e-6 for 3x3 layers through F(2x2,3x3), 1.5e-6
    # after a whole U-Net, 0.04e-6 for the elementwise optimizer step.  Two
    # correct orders of summation differ by up to twice that; four to six
    # times it is allowed.
    return {"rel": 5e-7 if case["kind"] == "adamw" else 1e-5}
