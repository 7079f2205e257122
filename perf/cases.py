"""The library's performance cases: what a program that renders with it has it
do, operation by operation, plus one whole UNet step.

`listed()` names the cases, `draw(rng)` gives others of the same ranges,
`prepare(case, seed)` makes what such a program holds before the call (tensors
on the GPU, their descriptors, the chain, the work buffer; for the two graphs,
the model and its captured graph), `run(state)` is one pass through the public
entry points, `work(case)` the bytes and operations that the pass cannot do
without, `tolerance(case)` how far two correct implementations may differ, and
`exact(case, seed)` the same outputs in 64-bit torch.

Sizes are those of SD1.5's UNet at 512x512 and around, of its VAE decoder, and
of SDXL's transformer block (bench.py), with images that are not square among
them: 520 x 768 pixels is a latent of 65 x 96, whose levels are 65 x 96,
33 x 48 and 17 x 24 tokens.
"""

import ctypes
import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "stable-diffusion.assembly_amd"))

import sdhip  # noqa: E402
import unet_step  # noqa: E402

SDXL_TUNING = "bits=8,weight_group=0"
GELU_K = 2.0 * math.sqrt(2.0 / math.pi)


def listed():
    return [
        # The keys (or values) of one cross-attention: the prompt's 77 tokens,
        # twice for guidance, to the first level's 320 channels.  The smallest
        # call, of which a step has 32.
        dict(name="linear context", kind="linear", batch=2, tokens=77, inner=768, outer=320, bias=False),
        # A projection at the first level of a 512x512 image, with its bias.
        dict(name="linear 320", kind="linear", batch=2, tokens=4096, inner=320, outer=320, bias=True),
        # LayerNorm, the gated feed-forward and its way back with bias and
        # residual, at the second level of a 520x768 image.
        dict(name="feed forward", kind="feed_forward", batch=2, tokens=33 * 48, channels=640),
        # The ResBlock's 3x3 convolution at the first level with bias and
        # residual: the headline of bench.py.
        dict(name="conv3x3 320 64x64", kind="conv", batch=2, inner=320, outer=320, height=64, width=64, size=3,
             residual=True, norm=False),
        # The ResBlock's 3x3 convolution at the lowest level, then GROUP_NORM
        # and SiLU: bound by its 29.5 MB of weights.
        dict(name="conv3x3 1280 8x8", kind="conv", batch=2, inner=1280, outer=1280, height=8, width=8, size=3,
             residual=False, norm=True),
        # The VAE decoder's last level at full size: the largest single convolution.
        dict(name="conv3x3 128 520x768", kind="conv", batch=1, inner=128, outer=128, height=520, width=768, size=3,
             residual=True, norm=False),
        # A 1x1 convolution (a ResBlock's skip), then GROUP_NORM and SiLU.
        dict(name="conv1x1 640-1280 32x32", kind="conv", batch=2, inner=640, outer=1280, height=32, width=32, size=1,
             residual=False, norm=True),
        # Self-attention at the first level of a 512x512 image.
        dict(name="attention 4096x40", kind="attention", batch=2, heads=8, queries=4096, keys=4096, dim=40),
        # Cross-attention to the prompt at the first level of a 520x768 image.
        dict(name="attention 77 keys", kind="attention", batch=2, heads=8, queries=65 * 96, keys=77, dim=40),
        # The VAE's middle attention: one head of 512.
        dict(name="attention 4096x512", kind="attention", batch=1, heads=1, queries=4096, keys=4096, dim=512),
        # SDXL's transformer block with int8 products (bits=8), quantized
        # weights kept in the store, replayed from a captured graph.
        dict(name="sdxl block bits=8", kind="sdxl_block", batch=2, tokens=988, channels=1280, heads=20),
        # One denoising step of SD1.5's UNet at 512x512 with guidance,
        # replayed from a captured graph: the whole call of a sampler.
        dict(name="unet step", kind="unet", batch=2, latent=64),
    ]


def _log_int(rng, low, high, multiple=1):
    """An integer spread over the logarithm of [low, high], a multiple of `multiple`."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / multiple)) * multiple))


def draw(rng):
    kind = rng.choice(["linear", "feed_forward", "conv3", "conv3", "conv1", "self", "cross", "vae attention",
                       "sdxl_block", "unet"])
    batch = rng.choice([1, 2])
    # A level of the UNet (the lowest has convolutions only): its channels,
    # and its image for 384 .. 768 pixels a side.
    level = rng.randrange(4 if kind in ("conv3", "conv1") else 3)
    channels = 320 << min(level, 2)
    height, width = (-(-rng.randint(48, 96) // (1 << level)) for _ in range(2))
    if kind == "linear":
        return dict(kind="linear", batch=batch, tokens=_log_int(rng, 64, 9216), inner=rng.choice([320, 640, 768, 1280]),
                    outer=rng.choice([320, 640, 1280]), bias=rng.random() < 0.5)
    if kind == "feed_forward":
        return dict(kind="feed_forward", batch=batch, tokens=height * width, channels=channels)
    if kind == "conv3" and rng.random() < 0.4:
        # The VAE's levels: 512, 256 or 128 channels.
        c = rng.choice([128, 256, 512])
        most = 65536 // c
        return dict(kind="conv", batch=1, inner=c, outer=c, height=_log_int(rng, 64, most), width=_log_int(rng, 64, most),
                    size=3, residual=rng.random() < 0.5, norm=False)
    if kind in ("conv3", "conv1"):
        # The UNet's: the inputs of the way up are two maps side by side.
        return dict(kind="conv", batch=batch, inner=channels * rng.choice([1, 2]), outer=channels, height=height,
                    width=width, size=3 if kind == "conv3" else 1, residual=rng.random() < 0.5,
                    norm=rng.random() < 0.5)
    if kind == "self":
        return dict(kind="attention", batch=batch, heads=8, queries=height * width, keys=height * width, dim=channels // 8)
    if kind == "cross":
        return dict(kind="attention", batch=batch, heads=8, queries=height * width, keys=rng.choice([77, 154]),
                    dim=channels // 8)
    if kind == "vae attention":
        tokens = _log_int(rng, 1024, 6144)
        return dict(kind="attention", batch=1, heads=1, queries=tokens, keys=tokens, dim=512)
    if kind == "sdxl_block":
        return dict(kind="sdxl_block", batch=batch, tokens=_log_int(rng, 512, 2048), channels=1280, heads=20)
    return dict(kind="unet", batch=batch, latent=8 * rng.randint(3, 8))


# ---------------------------------------------------------------- inputs


class _Source:
    """Activations ~N(0, 1), FP16 weights ~N(0, 0.02), biases ~N(0, 0.01) and
    norms ~N(1, 0.1), N(0, 0.1), on the GPU, from a seed alone."""

    def __init__(self, seed):
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.device).manual_seed(seed)

    def values(self, *shape, std=1.0, mean=0.0):
        return mean + std * torch.randn(shape, generator=self.gen, device=self.device)

    def weights(self, *shape):
        return self.values(*shape, std=0.02).to(torch.float16)


def _inputs(case, seed):
    """The case's tensors by name."""
    src = _Source(seed)
    kind = case["kind"]
    if kind == "linear":
        t = dict(x=src.values(case["batch"], case["tokens"], case["inner"]),
                 w=src.weights(case["outer"], case["inner"]))
        if case["bias"]:
            t["bias"] = src.values(case["outer"], std=0.01)
        return t
    if kind == "feed_forward":
        c = case["channels"]
        return dict(x=src.values(case["batch"], case["tokens"], c), gamma=src.values(c, std=0.1, mean=1.0),
                    beta=src.values(c, std=0.1), w1=src.weights(8 * c, c), b1=src.values(8 * c, std=0.01),
                    w2=src.weights(c, 4 * c), b2=src.values(c, std=0.01))
    if kind == "conv":
        oc, k = case["outer"], case["size"]
        t = dict(x=src.values(case["batch"], case["inner"], case["height"], case["width"]),
                 w=src.weights(oc, case["inner"], k, k), bias=src.values(1, oc, 1, 1, std=0.01))
        if case["residual"]:
            t["residual"] = src.values(case["batch"], oc, case["height"], case["width"])
        if case["norm"]:
            t.update(gamma=src.values(1, oc, 1, 1, std=0.1, mean=1.0), beta=src.values(1, oc, 1, 1, std=0.1))
        return t
    if kind == "attention":
        b, h, d = case["batch"], case["heads"], case["dim"]
        return dict(q=src.values(b, case["queries"], h, d), k=src.values(b, case["keys"], h, d),
                    v=src.values(b, case["keys"], h, d))
    if kind == "sdxl_block":
        block = unet_step.SdxlBlock(src.device, channels=case["channels"], heads=case["heads"], seed=seed)
        return dict(block=block, x=src.values(case["batch"], case["tokens"], case["channels"]))
    model = unet_step.Model(unet_step.Config(batch=case["batch"], latent=case["latent"]), src.device, seed=seed)
    x, t, context = model.inputs(seed=seed + 1)
    return dict(model=model, x=x, t=t, context=context)


# ---------------------------------------------------------------- the passes


class _Calls:
    """The library's calls of a pass, their descriptors, chains and work
    buffers made once, as a program with a fixed graph keeps them."""

    def __init__(self, tensors):
        self.lib = sdhip.load()
        sdhip.check(self.lib.sdhip_init(torch.cuda.current_device()), "init")
        self.tensors = tensors
        self.calls = []
        self.held = []
        self.out = None

    def _chain(self, steps):
        if not steps:
            return None
        chain = sdhip.epilogue(steps)
        self.held.append(chain)
        return ctypes.byref(chain)

    def _work(self, size):
        buf = torch.empty(max(size, 16), dtype=torch.uint8, device="cuda")
        self.held.append(buf)
        return ctypes.c_void_p(buf.data_ptr()), ctypes.c_size_t(size)

    def _keep(self, y, *tensors):
        """The output and the descriptors of a call; what they point at is held."""
        self.held += list(tensors)
        self.out = y
        return [sdhip.desc(t) for t in tensors]

    def linear(self, x, w, steps):
        y = torch.empty((*x.shape[:-1], w.shape[0]), device=x.device)
        dw, dx, dy = self._keep(y, w, x, y)
        work = self._work(self.lib.sdhip_mul_mat_work_size(dw, dx, dy))
        self.calls.append((self.lib.sdhip_mul_mat, (dw, dx, dy, self._chain(steps), *work)))
        return y

    def geglu(self, x, w, steps):
        y = torch.empty((*x.shape[:-1], w.shape[0]), device=x.device)  # described, never written
        out = torch.empty((*x.shape[:-1], w.shape[0] // 2), device=x.device)
        dw, dx, dy, do = self._keep(out, w, x, y, out)
        work = self._work(self.lib.sdhip_mul_mat_work_size(dw, dx, dy))
        self.calls.append((self.lib.sdhip_mul_mat_gated, (dw, dx, dy, self._chain(steps), do, *work)))
        return out

    def layer_norm(self, x, gamma, beta):
        y = torch.empty_like(x)
        dx, dy = self._keep(y, x, y)
        self.calls.append((self.lib.sdhip_norm, (dx, dy, 1e-5, self._chain([("mul", gamma), ("add", beta)]))))
        return y

    def group_norm(self, x, gamma, beta):
        y = torch.empty_like(x)
        dx, dy = self._keep(y, x, y)
        work = self._work(self.lib.sdhip_group_norm_work_size(dx, dy, 32))
        chain = self._chain([("mul", gamma), ("add", beta), ("silu", None)])
        self.calls.append((self.lib.sdhip_group_norm, (dx, dy, 32, 1e-5, chain, *work)))
        return y

    def conv(self, x, w, steps):
        pad = w.shape[2] // 2
        y = torch.empty((x.shape[0], w.shape[0], x.shape[2], x.shape[3]), device=x.device)
        params = sdhip.conv_params(1, 1, pad, pad, 1, 1)
        dw, dx, dy = self._keep(y, w, x, y)
        work = self._work(self.lib.sdhip_conv2d_work_size(dw, dx, dy, params))
        self.calls.append((self.lib.sdhip_conv2d, (dw, dx, dy, params, self._chain(steps), *work)))
        return y

    def attention(self, q, k, v):
        b, lq, h, d = q.shape
        y = torch.empty((b, lq, h, v.shape[3]), device=q.device)
        dq, dk, dv, dy = self._keep(y, *(t.permute(0, 2, 1, 3) for t in (q, k, v)), y)
        work = self._work(self.lib.sdhip_attention_work_size(dq, dk, dv, dy))
        self.calls.append((self.lib.sdhip_attention, (dq, dk, dv, dy, 1.0 / math.sqrt(d), 0.0, 0.0, *work)))
        return y

    def run(self):
        stream = sdhip.stream_handle()
        for fn, args in self.calls:
            sdhip.check(fn(*args, stream), fn.__name__)
        return self.out


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "sdxl_block":
        # A program in the bits mode sets its tuning and its store's arena
        # once; here they hold for the capture only, since both are the
        # process's and other cases run beside this one.
        sdhip.set_tuning(SDXL_TUNING)
        arena = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
        sdhip.store_arena(arena)
        ops = unet_step.HipOps(t["x"].device)
        try:
            graph = unet_step.Graph(lambda: t["block"].forward(ops, t["x"]), ops)
        finally:
            sdhip.store_arena(None)
            sdhip.set_tuning("")
        graph.held = (t, arena)
        return graph
    if kind == "unet":
        return unet_step.Step(t["model"], unet_step.HipOps(t["x"].device), (t["x"], t["t"], t["context"]))
    calls = _Calls(t)
    if kind == "linear":
        calls.linear(t["x"], t["w"], [("add", t["bias"])] if case["bias"] else [])
    elif kind == "feed_forward":
        h = calls.layer_norm(t["x"], t["gamma"], t["beta"])
        h = calls.geglu(h, t["w1"], [("add", t["b1"])])
        calls.linear(h, t["w2"], [("add", t["b2"]), ("add", t["x"])])
    elif kind == "conv":
        h = calls.conv(t["x"], t["w"], [("add", t["bias"])] + ([("add", t["residual"])] if case["residual"] else []))
        if case["norm"]:
            calls.group_norm(h, t["gamma"], t["beta"])
    else:
        calls.attention(t["q"], t["k"], t["v"])
    return calls


def run(state):
    return state.run()


# ---------------------------------------------------------------- what a pass cannot do without


def _unet_work(case):
    """Floating-point operations of the nodes, and the weights, inputs and
    output once each, counted on tensors without storage."""
    model = unet_step.Model(unet_step.Config(batch=case["batch"], latent=case["latent"]), "meta")
    ops = unet_step.TorchOps(torch.float32)
    x = torch.empty((case["batch"], 4, case["latent"], case["latent"]), device="meta")
    context = torch.empty((case["batch"], 77, 768), device="meta")
    model.forward(ops, x, torch.empty(case["batch"], device="meta"), context)

    def size(o):
        if isinstance(o, torch.Tensor):
            return o.numel() * o.element_size()
        if isinstance(o, dict):
            return sum(size(v) for v in o.values())
        return sum(size(v) for v in o) if isinstance(o, (list, tuple)) else 0

    weights = sum(size(getattr(model, n)) for n in ("time", "conv_in", "down", "mid", "up", "out_norm", "conv_out"))
    return dict(bytes=weights + 4 * (2 * x.numel() + context.numel()), flops=ops.flops)


def work(case):
    kind = case["kind"]
    if kind == "unet":
        return _unet_work(case)
    if kind == "linear":
        m, k, n = case["batch"] * case["tokens"], case["inner"], case["outer"]
        return dict(bytes=4 * m * k + 2 * k * n + 4 * m * n, flops=2 * m * k * n)
    if kind == "feed_forward":
        m, c = case["batch"] * case["tokens"], case["channels"]
        return dict(bytes=8 * m * c + 24 * c * c, flops=24 * m * c * c)
    if kind == "sdxl_block":
        b, l, c = case["batch"], case["tokens"], case["channels"]
        return dict(bytes=8 * b * l * c + 16 * c * c, flops=2 * b * l * 16 * c * c + 4 * b * l * l * c)
    if kind == "conv":
        ic, oc, k = case["inner"], case["outer"], case["size"]
        p = case["batch"] * case["height"] * case["width"]
        return dict(bytes=4 * p * (ic + oc * (2 if case["residual"] else 1)) + 2 * ic * oc * k * k,
                    flops=2 * p * ic * oc * k * k)
    b, h, lq, lk, d = (case[n] for n in ("batch", "heads", "queries", "keys", "dim"))
    return dict(bytes=8 * b * h * d * (lq + lk), flops=4 * b * h * lq * lk * d)


def tolerance(case):
    # Single precision throughout, sums in any order: 1e-5 (operations measure
    # 3e-7 .. 1.1e-6 from 64 bits).  A whole step: inputs changed in their
    # last bit move its output by 4.6e-6.  The block in int8: the same change
    # of its inputs moves its output by 1.7e-3, where roundings to 8 bits
    # fall the other way.
    return {"rel": {"sdxl_block": 7e-3, "unet": 2e-5}.get(case["kind"], 1e-5)}


# ---------------------------------------------------------------- 64 bits


def _linear64(x, w, bias=None):
    y = x @ w.double().t()
    return y if bias is None else y + bias.double()


def _geglu64(x, w, bias):
    a, g = _linear64(x, w, bias).chunk(2, dim=-1)
    return a * (g / (1.0 + torch.exp(-GELU_K * g * (1.0 + 0.044715 * g * g))))


def _layer_norm64(x, gamma, beta):
    return F.layer_norm(x, (x.shape[-1],), gamma.double(), beta.double(), 1e-5)


def _group_norm64(x, gamma, beta, eps=1e-5, silu=True):
    y = F.group_norm(x, 32, gamma.double().reshape(-1), beta.double().reshape(-1), eps)
    return F.silu(y) if silu else y


def _conv64(x, w, bias, stride=1):
    """By columns of one image at a time: a product for each tap."""
    w = w.double()
    k = w.shape[2]
    pad = k // 2
    xp = F.pad(x.double(), (pad,) * 4)
    oh, ow = ((s + 2 * pad - k) // stride + 1 for s in x.shape[2:])
    out = []
    for image in xp:
        y = 0.0
        for i in range(k):
            for j in range(k):
                part = image[:, i:i + stride * (oh - 1) + 1:stride, j:j + stride * (ow - 1) + 1:stride]
                y = y + w[:, :, i, j].contiguous() @ part.reshape(part.shape[0], -1)
        out.append(y.view(-1, oh, ow))
    return torch.stack(out) + bias.double().reshape(1, -1, 1, 1)


def _attention64(q, k, v):
    """[b, l, h, d] each, a head at a time."""
    out = torch.empty((*q.shape[:3], v.shape[3]), dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            s = q[b, :, h].double() @ k[b, :, h].double().t().contiguous() / math.sqrt(q.shape[3])
            out[b, :, h] = torch.softmax(s, dim=-1) @ v[b, :, h].double()
    return out


def _heads64(q, k, v, heads):
    split = [t.view(t.shape[0], t.shape[1], heads, -1) for t in (q, k, v)]
    return _attention64(*split).view(q.shape)


def _sdxl64(block, x):
    x = x.double()
    n = _layer_norm64(x, *block.ln1)
    q, k, v = (_linear64(n, w) for w in (block.wq, block.wk, block.wv))
    x = x + _linear64(_heads64(q, k, v, block.heads), *block.wo)
    return x + _linear64(_geglu64(_layer_norm64(x, *block.ln2), *block.ff1), *block.ff2)


def _resblock64(p, x, projections):
    h = _group_norm64(x, *p["norm1"])
    h = _conv64(h, *p["conv1"]) + projections[p["emb_at"]][:, :, None, None]
    h = _conv64(_group_norm64(h, *p["norm2"]), *p["conv2"])
    return h + (x if p["skip"] is None else _conv64(x, *p["skip"]))


def _transformer64(p, x, context, heads):
    b, c, hh, ww = x.shape
    h = _conv64(_group_norm64(x, *p["norm"], eps=1e-6, silu=False), *p["proj_in"])
    t = h.flatten(2).transpose(1, 2).contiguous()
    n = _layer_norm64(t, *p["ln1"])
    t = t + _linear64(_heads64(*(_linear64(n, p[w][0]) for w in ("q1", "k1", "v1")), heads), *p["o1"])
    q = _linear64(_layer_norm64(t, *p["ln2"]), p["q2"][0])
    t = t + _linear64(_heads64(q, *(_linear64(context, p[w][0]) for w in ("k2", "v2")), heads), *p["o2"])
    t = t + _linear64(_geglu64(_layer_norm64(t, *p["ln3"]), *p["ff1"]), *p["ff2"])
    return x + _conv64(t.transpose(1, 2).reshape(b, c, hh, ww), *p["proj_out"])


def _unet64(m, x, t, context):
    heads = m.cfg.heads
    half = m.cfg.channels // 2
    angles = t.double()[:, None] * torch.exp(
        -math.log(10000.0) * torch.arange(half, dtype=torch.float64, device=t.device) / half)
    # The embedding reaches the step in single precision.
    emb = torch.cat([angles.cos(), angles.sin()], dim=-1).float().double()
    emb = _linear64(F.silu(_linear64(emb, *m.time[0])), *m.time[1])
    projections = _linear64(F.silu(emb), *m.emb_all)
    context = context.double()
    h = _conv64(x, *m.conv_in)
    skips = [h]
    for blocks, down in m.down:
        for res, st in blocks:
            h = _resblock64(res, h, projections)
            if st is not None:
                h = _transformer64(st, h, context, heads)
            skips.append(h)
        if down is not None:
            h = _conv64(h, *down, stride=2)
            skips.append(h)
    res1, st, res2 = m.mid
    h = _resblock64(res1, h, projections)
    h = _resblock64(res2, _transformer64(st, h, context, heads), projections)
    for blocks, up in m.up:
        for res, st in blocks:
            h = _resblock64(res, torch.cat([h, skips.pop()], dim=1), projections)
            if st is not None:
                h = _transformer64(st, h, context, heads)
        if up is not None:
            h = _conv64(F.interpolate(h, scale_factor=2.0, mode="nearest"), *up)
    return _conv64(_group_norm64(h, *m.out_norm), *m.conv_out)


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return _linear64(t["x"].double(), t["w"], t.get("bias"))
    if kind == "feed_forward":
        x = t["x"].double()
        h = _geglu64(_layer_norm64(x, t["gamma"], t["beta"]), t["w1"], t["b1"])
        return _linear64(h, t["w2"], t["b2"]) + x
    if kind == "conv":
        y = _conv64(t["x"], t["w"], t["bias"])
        y = y + t["residual"] if case["residual"] else y
        return _group_norm64(y, t["gamma"], t["beta"]) if case["norm"] else y
    if kind == "attention":
        return _attention64(t["q"], t["k"], t["v"])
    if kind == "sdxl_block":
        return _sdxl64(t["block"], t["x"])
    return _unet64(t["model"], t["x"], t["t"], t["context"])
