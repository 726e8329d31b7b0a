"""The workloads whose speed this library is judged by: inputs, one pass through
the public entry points, the work it cannot do without, and the same results in
64 bits by plain torch.

Every case is a dict of plain values; ``kind`` selects the path:

``conv``    Conv2d, fwd (``train`` false) or fwd + dX + dW + db
``convt``   ConvTranspose2d, fwd + dX + dW + db
``linear``  Linear, fwd + dX + dW + db
``matmul``  gpu_matmul and its two gradients
``chain``   a ConvChain training step: conv / ReLU layers, an optional PixelShuffle,
            sum loss, seeded backward
"""
import torch
import torch.nn.functional as F

from volta_amd import nn, ops

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _conv(n, c, o, h, w, k, s, p, dtype, train=True):
    return dict(kind="conv", n=n, c=c, o=o, h=h, w=w, k=k, s=s, p=p, dtype=dtype, train=train)


def listed():
    def named(name, case):
        return dict(case, name=name)

    return [
        # one image through one layer: serving at batch 1, where latency is everything
        named("conv3x3_infer_bf16", _conv(1, 64, 64, 56, 56, 3, 1, 1, "bf16", train=False)),
        # the middle layer of the ResNet-style block that the benchmark is quoted on
        named("conv3x3_train_bf16", _conv(128, 128, 128, 28, 28, 3, 1, 1, "bf16")),
        # images cropped to no particular size, channel counts off the tile sizes
        named("conv3x3_train_bf16_odd", _conv(32, 96, 144, 35, 27, 3, 1, 1, "bf16")),
        # a down-sampling layer between two stages of a residual network
        named("conv3x3s2_train_bf16", _conv(64, 64, 128, 56, 56, 3, 2, 1, "bf16")),
        # the library's default dtype: a layer of a network for 32 x 32 images
        named("conv3x3_train_f32", _conv(64, 64, 128, 32, 32, 3, 1, 1, "f32")),
        # a generator's up-sampling layer (DCGAN, 8 x 8 -> 16 x 16)
        named("convt4x4s2_train_f32", dict(kind="convt", n=128, c=256, o=128, h=8, w=8, k=4, s=2, p=1, dtype="f32")),
        # the first layer of an MLP over flattened 28 x 28 images
        named("linear_train_f32", dict(kind="linear", m=256, i=784, o=512, dtype="f32")),
        # the Linear benchmark: 4096 rows, 1024 -> 4096
        named("linear_train_bf16", dict(kind="linear", m=4096, i=1024, o=4096, dtype="bf16")),
        # products whose sizes fit no tile, forward and both gradients
        named("matmul_bf16_odd", dict(kind="matmul", m=1500, k=2001, n=1111, dtype="bf16")),
        # a large product in the default dtype
        named("matmul_f32", dict(kind="matmul", m=2048, k=2048, n=2048, dtype="f32")),
        # the MNIST CNN training step: small layers, many launches
        named("mnist_cnn_step_f32", dict(kind="chain", net="mnist", n=64, h=28, w=28, dtype="f32")),
        # the super-resolution training step at 256 x 256: the largest
        named("sr_chain_step_bf16", dict(kind="chain", net="sr", n=16, h=256, w=256, dtype="bf16")),
    ]


def _log(rng, lo, hi):
    """An integer of lo .. hi, uniform over its logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def _channels(rng, lo, hi):
    """Two thirds of real layers' channel counts are multiples of 16; the rest is any number."""
    c = _log(rng, lo, hi)
    return c if rng.random() < 1 / 3 else max(16, (c + 8) // 16 * 16)


def _draw(rng):
    kind = rng.choice(["infer", "conv_bf16", "conv_bf16", "down_bf16", "conv_f32", "convt", "linear", "matmul",
                       "mnist", "sr"])
    if kind == "infer":
        h = _log(rng, 14, 112)
        return _conv(_log(rng, 1, 8), _channels(rng, 16, 256), _channels(rng, 16, 256), h,
                     h if rng.random() < 0.5 else _log(rng, 14, 112), 3, 1, 1, "bf16", train=False)
    if kind in ("conv_bf16", "down_bf16", "conv_f32"):
        k = rng.choice([1, 3, 3, 3, 5]) if kind != "down_bf16" else rng.choice([1, 3, 3])
        s = 2 if kind == "down_bf16" else 1
        h = _log(rng, 7, 64)
        return _conv(_log(rng, 4, 128), _channels(rng, 16, 256), _channels(rng, 16, 256), h,
                     h if rng.random() < 0.5 else _log(rng, 7, 64), k, s, k // 2,
                     "f32" if kind == "conv_f32" else "bf16")
    if kind == "convt":
        h = _log(rng, 4, 32)
        return dict(kind="convt", n=_log(rng, 4, 128), c=_channels(rng, 32, 512), o=_channels(rng, 16, 256), h=h,
                    w=h, k=4, s=2, p=1, dtype="f32")
    if kind == "linear":
        return dict(kind="linear", m=_log(rng, 32, 4096), i=_log(rng, 64, 4096), o=_log(rng, 64, 4096),
                    dtype=rng.choice(["f32", "bf16"]))
    if kind == "matmul":
        return dict(kind="matmul", m=_log(rng, 64, 8192), k=_log(rng, 64, 8192), n=_log(rng, 64, 8192),
                    dtype=rng.choice(["f32", "bf16"]))
    if kind == "mnist":
        return dict(kind="chain", net="mnist", n=_log(rng, 8, 256), h=28, w=28, dtype="f32")
    return dict(kind="chain", net="sr", n=_log(rng, 1, 16), h=_log(rng, 32, 255), w=_log(rng, 32, 255), dtype="bf16")


def draw(rng):
    limit = {("conv", "bf16"): 1.2e11, ("conv", "f32"): 3e10, ("convt", "f32"): 3e10, ("linear", "f32"): 5.2e10,
             ("matmul", "f32"): 5.2e10}
    while True:
        case = _draw(rng)
        if work(case)["flops"] <= limit.get((case["kind"], case["dtype"]), 4e11):
            return case


# ------------------------------------------------------------------ inputs
def _chain_specs(net):
    if net == "mnist":
        return [(1, 32, 3, 1, 1), (32, 64, 3, 1, 1)]
    return [(3, 64, 5, 1, 2), (64, 64, 3, 1, 1), (64, 32, 3, 1, 1), (32, 27, 3, 1, 1)]


def _inputs(case, seed):
    """The tensors of a case in its dtype, on the GPU: activations and output
    gradients N(0, 1) (chain inputs U[0, 1), as images are), He- or
    Xavier-scaled weights, small biases."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def normal(*shape, std=1.0):
        return (torch.randn(shape, generator=g, device=DEV) * std).to(dt)

    kind = case["kind"]
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(a=normal(m, k), b=normal(k, n), g=normal(m, n))
    if kind == "linear":
        m, i, o = case["m"], case["i"], case["o"]
        return dict(x=normal(m, i), w=normal(i, o, std=(2.0 / (i + o)) ** 0.5), b=normal(o, std=0.1), dy=normal(m, o))
    if kind == "chain":
        specs = _chain_specs(case["net"])
        x = torch.rand((case["n"], specs[0][0], case["h"], case["w"]), generator=g, device=DEV).to(dt)
        return dict(x=x, w=[normal(o, c, k, k, std=(2.0 / (c * k * k)) ** 0.5) for c, o, k, _, _ in specs],
                    b=[normal(o, std=0.1) for _, o, _, _, _ in specs])
    n, c, o, h, w, k, s, p = (case[f] for f in ("n", "c", "o", "h", "w", "k", "s", "p"))
    if kind == "convt":
        ho, wo = (h - 1) * s + k - 2 * p, (w - 1) * s + k - 2 * p
        weight = normal(c, o, k, k, std=(2.0 / (c * k * k)) ** 0.5)
    else:
        ho, wo = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
        weight = normal(o, c, k, k, std=(2.0 / (c * k * k)) ** 0.5)
    t = dict(x=normal(n, c, h, w), w=weight, b=normal(o, std=0.1))
    if case.get("train", True):
        t["dy"] = normal(n, o, ho, wo)
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    dt = DTYPES[case["dtype"]]
    kind = case["kind"]
    if kind == "matmul":
        return dict(t, dims=(case["m"], case["k"], case["n"]), kind=kind)
    if kind == "chain":
        chain = nn.ConvChain(_chain_specs(case["net"]), t["x"], tail=nn.PixelShuffle(3) if case["net"] == "sr" else None)
        for conv, w, b in zip(chain.convs, t["w"], t["b"]):
            conv.weight, conv.bias = w, b
        return dict(chain=chain, kind=kind)
    if kind == "linear":
        layer = nn.Linear(case["i"], case["o"], device=DEV, dtype=dt)
    else:
        cls = nn.Conv2d if kind == "conv" else nn.ConvTranspose2d
        layer = cls(case["c"], case["o"], case["k"], case["s"], case["p"], device=DEV, dtype=dt)
    layer.weight, layer.bias = t["w"], t["b"]
    return dict(layer=layer, x=t["x"], dy=t.get("dy"), kind=kind)


# ------------------------------------------------------------------ one pass
def run(state):
    if state["kind"] == "matmul":
        a, b, g, dims = state["a"], state["b"], state["g"], state["dims"]
        return ops.gpu_matmul(a, b, *dims), ops.gpu_matmul_backward_a(g, b, *dims), ops.gpu_matmul_backward_b(a, g, *dims)
    if state["kind"] == "chain":
        chain = state["chain"]
        chain.step()
        # the inner gradients stay out: where rounding moves a ReLU's input across zero, single values of them
        # come or go whole; the weight gradients hold what they add up to
        return [chain.loss, chain.output] + [t for pair in chain.wgrads for t in pair]
    layer, x, dy = state["layer"], state["x"], state["dy"]
    y = layer.forward(x)
    return y if dy is None else (y,) + tuple(layer.backward(dy, x))


# ------------------------------------------------------------------ what a pass cannot do without
def _conv_macs(n, c, o, k, ho, wo):
    return n * c * o * k * k * ho * wo


def work(case):
    es = 4 if case["dtype"] == "f32" else 2
    kind = case["kind"]
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": es * (2 * m * k + 2 * k * n + 2 * m * n), "flops": 6 * m * k * n}
    if kind == "linear":
        m, i, o = case["m"], case["i"], case["o"]
        return {"bytes": es * (2 * m * i + 2 * i * o + 2 * o + 2 * m * o), "flops": 6 * m * i * o}
    if kind == "chain":
        n, h, w = case["n"], case["h"], case["w"]
        specs = _chain_specs(case["net"])
        macs = weights = 0
        for l, (c, o, k, _, _) in enumerate(specs):
            macs += _conv_macs(n, c, o, k, h, w) * (3 if l else 2)  # the graph input needs no gradient
            weights += o * c * k * k + o
        # forward: every activation written once and read by the next layer; backward: every activation
        # read again, every gradient written and read (its seed is a constant)
        px = n * h * w
        outs = [o for _, o, _, _, _ in specs]
        elems = px * (2 * specs[0][0] + 3 * sum(outs[:-1]) + 2 * sum(outs[:-1]) + 2 * outs[-1]) + 2 * weights
        return {"bytes": es * elems, "flops": 2 * macs}
    n, c, o, h, w, k, s, p = (case[f] for f in ("n", "c", "o", "h", "w", "k", "s", "p"))
    if kind == "convt":
        ho, wo = (h - 1) * s + k - 2 * p, (w - 1) * s + k - 2 * p
        macs = _conv_macs(n, c, o, k, h, w)
    else:
        ho, wo = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
        macs = _conv_macs(n, c, o, k, ho, wo)
    x, y, wt = n * c * h * w, n * o * ho * wo, c * o * k * k + o
    if case.get("train", True):
        return {"bytes": es * 2 * (x + y + wt), "flops": 6 * macs}
    return {"bytes": es * (x + y + wt), "flops": 2 * macs}


def tolerance(case):
    """About four times what the specialised and the generic kernels of this
    library, which sum in different orders, differ by: single layers in bf16 up
    to 3e-5 (results rounded the other way: one unit of 2^-7 at most each), in
    f32 4e-7 at sums of 288 terms and 1.1e-6 at 2048 (two results each up to
    8e-7 off the 64-bit one); chains 3.6e-7 in f32 and 3.3e-4 in bf16, where a
    rounding travels through the layers that follow."""
    if case["dtype"] == "f32":
        return {"rel": 2e-6, "max": 4e-5} if case["kind"] == "chain" else {"rel": 5e-6, "max": 2e-4}
    return {"rel": 1.5e-3, "max": 0.05} if case["kind"] == "chain" else {"rel": 3e-4, "max": 0.02}


# ------------------------------------------------------------------ the same in 64 bits
def _patch(xp, r, q, s, ho, wo):
    """The input values that tap (r, q) reads, as a [C, N * ho * wo] matrix."""
    v = xp[:, :, r:r + s * (ho - 1) + 1:s, q:q + s * (wo - 1) + 1:s]
    return v.permute(1, 0, 2, 3).reshape(xp.shape[1], -1)


def _conv64(x, w, s, p):
    n, _, h, wd = x.shape
    o, _, k, _ = w.shape
    ho, wo = (h + 2 * p - k) // s + 1, (wd + 2 * p - k) // s + 1
    xp = F.pad(x, (p, p, p, p))
    y = torch.zeros((o, n * ho * wo), dtype=x.dtype, device=x.device)
    for r in range(k):
        for q in range(k):
            y += w[:, :, r, q] @ _patch(xp, r, q, s, ho, wo)
    return y.reshape(o, n, ho, wo).permute(1, 0, 2, 3).contiguous()


def _conv64_dx(dy, w, shape, s, p):
    n, c, h, wd = shape
    o, _, k, _ = w.shape
    ho, wo = dy.shape[2:]
    d = dy.permute(1, 0, 2, 3).reshape(o, -1)
    dxp = torch.zeros((n, c, h + 2 * p, wd + 2 * p), dtype=dy.dtype, device=dy.device)
    for r in range(k):
        for q in range(k):
            t = (w[:, :, r, q].t().contiguous() @ d).reshape(c, n, ho, wo).permute(1, 0, 2, 3)
            dxp[:, :, r:r + s * (ho - 1) + 1:s, q:q + s * (wo - 1) + 1:s] += t
    return dxp[:, :, p:p + h, p:p + wd].contiguous()


def _conv64_dw(dy, x, wshape, s, p):
    o, _, k, _ = wshape
    ho, wo = dy.shape[2:]
    d = dy.permute(1, 0, 2, 3).reshape(o, -1)
    xp = F.pad(x, (p, p, p, p))
    dw = torch.empty(wshape, dtype=dy.dtype, device=dy.device)
    for r in range(k):
        for q in range(k):
            dw[:, :, r, q] = d @ _patch(xp, r, q, s, ho, wo).t().contiguous()
    return dw


def _exact_chain(case, t):
    specs = _chain_specs(case["net"])
    acts = [t["x"]]
    for l, (w, b) in enumerate(zip(t["w"], t["b"])):
        y = _conv64(acts[-1], w, 1, specs[l][4]) + b[None, :, None, None]
        acts.append(y.clamp_min(0) if l + 1 < len(specs) else y)
    out = F.pixel_shuffle(acts[-1], 3) if case["net"] == "sr" else acts[-1]
    grad, wgrads = torch.ones_like(acts[-1]), []
    for l in reversed(range(len(specs))):
        wgrads[:0] = [_conv64_dw(grad, acts[l], t["w"][l].shape, 1, specs[l][4]), grad.sum((0, 2, 3))]
        if l:
            grad = _conv64_dx(grad, t["w"][l], acts[l].shape, 1, specs[l][4]) * (acts[l] > 0)
    return [out.sum().reshape(1), out] + wgrads


def exact(case, seed):
    def wide(v):
        return [u.double() for u in v] if isinstance(v, list) else v.double()

    t = {name: wide(v) for name, v in _inputs(case, seed).items()}
    kind = case["kind"]
    if kind == "matmul":
        return t["a"] @ t["b"], t["g"] @ t["b"].t().contiguous(), t["a"].t().contiguous() @ t["g"]
    if kind == "linear":
        x, w, dy = t["x"], t["w"], t["dy"]
        return x @ w + t["b"], dy @ w.t().contiguous(), x.t().contiguous() @ dy, dy.sum(0)
    if kind == "chain":
        return _exact_chain(case, t)
    x, w, s, p = t["x"], t["w"], case["s"], case["p"]
    bias = t["b"][None, :, None, None]
    if kind == "convt":
        ho, wo = t["dy"].shape[2:]
        y = _conv64_dx(x, w, (case["n"], case["o"], ho, wo), s, p) + bias
        return y, _conv64(t["dy"], w, s, p), _conv64_dw(x, t["dy"], w.shape, s, p), t["dy"].sum((0, 2, 3))
    y = _conv64(x, w, s, p) + bias
    if not case["train"]:
        return y
    dy = t["dy"]
    return y, _conv64_dx(dy, w, x.shape, s, p), _conv64_dw(dy, x, w.shape, s, p), dy.sum((0, 2, 3))
