"""The work that a user of this framework has it do, as measurable cases.

Each case is one pass through a public entry point: the Converse2D layer (inference and training), the
registered operator, the per-sample data step, the ConverseBlocks and the models.  Sizes are those of
this repository's benchmark, tests and model defaults, and generic photo and patch sizes.

A case is a dict of plain values; its "kind" names the entry point:
  layer  util_converse.Converse2D under no_grad (transfer table kept by the library while the weights stand)
  train  util_converse.Converse2D forward and all three gradients
  op     torch.ops.converse2d.forward(x, x0, weight, bias, scale, eps) under no_grad
  data   converse_usrnet.ConvReverseDataNet with a psf per sample (a new activation on every call)
  block  util_converse.ConverseBlock / ConverseBlockAlphaVariant under no_grad
  dncnn  converse_dncnn.ConverseDnCNN under no_grad
  usrnet converse_usrnet.ConverseUSRNet under no_grad
"""
import math

import torch
import torch.nn.functional as F

MODES = ("circular", "replicate", "reflect", "constant")


def _layer(name, kind, B, C, H, W, k, s, p, mode, eps=1e-5):
    c = {"kind": kind, "B": B, "C": C, "H": H, "W": W, "k": k, "s": s, "p": p, "mode": mode, "eps": eps}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one small feature map: latency, launches and host work count
        _layer("layer_small", "layer", 1, 64, 128, 128, 5, 1, 2, "circular"),
        # the headline layer: a batch of 256 x 256 feature maps
        _layer("layer_256", "layer", 16, 64, 256, 256, 5, 1, 2, "circular"),
        # a denoiser's layer on one photo of odd size (padded plane 333 x 493)
        _layer("layer_photo", "layer", 1, 128, 321, 481, 7, 1, 6, "circular"),
        # the super-resolution network's x2 upsampler (padded plane 132 -> 264)
        _layer("layer_up2", "layer", 4, 64, 128, 128, 2, 2, 2, "replicate", 1e-3),
        # the reference's operator timing grid at scale 3, x0 given by the caller
        {"name": "op_s3", "kind": "op", "B": 8, "C": 8, "H": 256, "W": 256, "k": 5, "s": 3, "eps": 1e-5},
        # a deblurring network's data step with a 25 x 25 psf per sample (the table is part of every call)
        {"name": "data_256", "kind": "data", "B": 4, "C": 64, "H": 256, "W": 256, "k": 25, "s": 1},
        # training: forward and all gradients of the headline layer
        _layer("train_256", "train", 16, 64, 256, 256, 5, 1, 2, "circular"),
        # training on 96 x 96 patches, the denoiser's layer (padded plane 108 x 108)
        _layer("train_patch", "train", 8, 128, 96, 96, 7, 1, 6, "circular"),
        # one block of the super-resolution body (padded plane 136 x 136)
        {"name": "block_sr", "kind": "block", "alpha": False, "B": 4, "C": 64, "H": 128, "W": 128, "k": 5, "p": 4,
         "mode": "replicate"},
        # one block of the denoiser's body at the benchmark's batch
        {"name": "block_dncnn", "kind": "block", "alpha": False, "B": 8, "C": 64, "H": 256, "W": 256, "k": 7, "p": 6,
         "mode": "circular"},
        # the denoiser on one photo of odd size, the evaluation loop's call
        {"name": "dncnn_photo", "kind": "dncnn", "B": 1, "H": 321, "W": 481},
        # the benchmark's super-resolution network: 4 images 64 x 64 -> 256 x 256, a 25 x 25 blur kernel each
        {"name": "usrnet_x4", "kind": "usrnet", "B": 4, "H": 64, "W": 64, "k": 25, "s": 4},
    ]


def _side(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, per_sample, budget, top):
    """A batch size, over its logarithm, that keeps the case within `budget` padded output samples."""
    return max(1, _side(rng, 1, max(1, min(top, budget // max(1, per_sample)))))


def draw(rng):
    kind = rng.choice(("layer",) * 5 + ("train",) * 3 + ("op", "op", "data", "data", "block", "block", "dncnn", "usrnet"))
    H = _side(rng, 24, 512)
    W = min(512, max(24, int(round(H * math.exp(rng.uniform(-0.5, 0.5))))))
    if kind == "layer":
        s = rng.choice((1, 1, 1, 2, 3, 4))
        H, W = max(16, H // s), max(16, W // s)
        k = rng.choice((2, 3, 4, 5, 7))
        p = rng.choice((0, 1, 2, 3, 4, 6))
        C = rng.choice((32, 64, 64, 128))
        B = _batch(rng, C * (H + 2 * p) * (W + 2 * p) * s * s, 40_000_000, 16)
        return _layer(None, kind, B, C, H, W, k, s, p, rng.choice(MODES), rng.choice((1e-5, 1e-3)))
    if kind == "train":
        s = rng.choice((1, 1, 2))
        H, W = max(16, H // (2 * s)), max(16, W // (2 * s))
        C = rng.choice((32, 64, 128))
        p = rng.choice((0, 1, 2, 4, 6))
        B = _batch(rng, C * (H + 2 * p) * (W + 2 * p) * s * s, 20_000_000, 16)
        return _layer(None, kind, B, C, H, W, rng.choice((2, 3, 5, 7)), s, p, rng.choice(MODES))
    if kind == "op":
        s = rng.choice((1, 2, 3, 4))
        H, W = max(16, H // s), max(16, W // s)
        C = rng.choice((8, 16, 64))
        return {"kind": "op", "B": _batch(rng, C * H * W * s * s, 30_000_000, 8), "C": C, "H": H, "W": W,
                "k": rng.choice((3, 5, 7)), "s": s, "eps": 1e-5}
    if kind == "data":
        s = rng.choice((1, 1, 2, 3, 4))
        H, W = max(16, H // s), max(16, W // s)
        return {"kind": "data", "B": _batch(rng, 64 * H * W * s * s, 17_000_000, 4), "C": 64, "H": H,
                "W": W, "k": min(rng.choice((7, 15, 25)), 2 * (min(H, W) * s // 2) - 1), "s": s}
    if kind == "block":
        p, k = rng.choice(((2, 3), (4, 5), (6, 7)))
        return {"kind": "block", "alpha": rng.random() < 0.5,
                "B": _batch(rng, 128 * (H + 2 * p) * (W + 2 * p), 40_000_000, 8), "C": 64, "H": H, "W": W, "k": k,
                "p": p, "mode": rng.choice(("circular", "replicate"))}
    if kind == "usrnet":
        s = rng.choice((2, 3, 4))
        H, W = min(80, max(16, H // s)), min(80, max(16, W // s))
        return {"kind": "usrnet", "B": _batch(rng, H * W * s * s, 200_000, 4), "H": H, "W": W,
                "k": rng.choice((7, 25)), "s": s}
    return {"kind": "dncnn", "B": 1, "H": min(H, 400), "W": min(W, 400)}


# --------------------------------------------------------------------------------------------------
# inputs and weights
# --------------------------------------------------------------------------------------------------
def _psf(g, n, C, k):
    """Softmax-normalised taps, as Converse2D initialises them."""
    return torch.softmax(torch.randn(n, C, k * k, device="cuda", generator=g), -1).view(n, C, k, k)


def _fill(m, g):
    """Weights of a network in use: fan-in-scaled layers, softmax psfs, norms near identity, small biases."""
    with torch.no_grad():
        for name, q in m.named_parameters():
            r = torch.randn(q.shape, device=q.device, generator=g)
            if q.dim() == 4 and q.shape[0] == 1 and q.shape[-1] > 1:
                q.copy_(_psf(g, 1, q.shape[1], q.shape[2]))
            elif "alpha" in name:
                q.copy_(0.3 * r)
            elif q.dim() >= 2 and q.shape[0] > 1:
                q.copy_(r / math.sqrt(q[0].numel()))
            elif name.endswith("weight"):
                q.copy_(1 + 0.1 * r)
            else:
                q.copy_(0.1 * r)
    return m


def _photo(g, B, ch, H, W):
    """Images in [0, 1]: a few smooth waves, and sensor noise."""
    y = torch.arange(H, device="cuda").view(1, 1, 1, H, 1) / H
    x = torch.arange(W, device="cuda").view(1, 1, 1, 1, W) / W
    f = torch.rand(3, B, ch, 6, 1, 1, device="cuda", generator=g)
    img = torch.sin(25 * (f[0] * y + f[1] * x) + 6.3 * f[2]).mean(2) * 0.4 + 0.5
    return img + torch.randn(img.shape, device="cuda", generator=g) * (25 / 255)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    c, kind = case, case["kind"]
    if kind == "dncnn":
        from conversenet_amd.converse_dncnn import ConverseDnCNN

        return {"case": c, "x": _photo(g, c["B"], 1, c["H"], c["W"]),
                "net": _fill(ConverseDnCNN().cuda().eval(), g)}
    if kind == "usrnet":
        from conversenet_amd.converse_usrnet import ConverseUSRNet

        k = torch.softmax(3 * torch.randn(c["B"], c["k"] ** 2, device="cuda", generator=g), -1)
        return {"case": c, "x": _photo(g, c["B"], 3, c["H"], c["W"]), "k": k.view(c["B"], 1, c["k"], c["k"]),
                "net": _fill(ConverseUSRNet(kernel_size=c["k"]).cuda().eval(), g)}
    B, C, H, W = c["B"], c["C"], c["H"], c["W"]
    x = torch.randn(B, C, H, W, device="cuda", generator=g)
    st = {"case": c, "x": x}
    if kind in ("layer", "train"):
        from conversenet_amd.util_converse import Converse2D

        m = Converse2D(C, C, c["k"], c["s"], c["p"], c["mode"], c["eps"]).cuda()
        with torch.no_grad():
            m.weight.copy_(_psf(g, 1, C, c["k"]))
            m.bias.copy_(0.3 * torch.randn(m.bias.shape, device="cuda", generator=g))
        st["net"] = m
        if kind == "train":
            x.requires_grad_(True)
            st["go"] = torch.randn(B, C, H * c["s"], W * c["s"], device="cuda", generator=g)
    elif kind == "op":
        import conversenet_amd  # noqa: F401  (registers the operator)

        st["x0"] = torch.randn(B, C, H * c["s"], W * c["s"], device="cuda", generator=g)
        st["w"] = _psf(g, 1, C, c["k"])
        st["b"] = 0.3 * torch.randn(1, C, 1, 1, device="cuda", generator=g)
    elif kind == "data":
        from conversenet_amd.converse_usrnet import ConvReverseDataNet

        m = ConvReverseDataNet().cuda()
        with torch.no_grad():
            m.alpha.copy_(0.3 * torch.randn(m.alpha.shape, device="cuda", generator=g))
        st["net"] = m
        st["k"] = _psf(g, B, C, c["k"])
    else:
        from conversenet_amd import util_converse as U

        cls = U.ConverseBlockAlphaVariant if c["alpha"] else U.ConverseBlock
        st["net"] = _fill(cls(C, C, c["k"], 1, c["p"], c["mode"], 1e-5).cuda().eval(), g)
    return st


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "train":
        m, x = state["net"], state["x"]
        out = m(x)
        gx, gw, gb = torch.autograd.grad(out, (x, m.weight, m.bias), state["go"])
        return {"out": out.detach(), "gx": gx, "gw": gw, "gb": gb}
    with torch.no_grad():
        if kind == "op":
            return torch.ops.converse2d.forward(state["x"], state["x0"], state["w"], state["b"], c["s"], c["eps"])
        if kind == "data":
            return state["net"](state["x"], state["k"], c["s"])
        if kind == "usrnet":
            return state["net"](state["x"], state["k"], c["s"])
        return state["net"](state["x"])


# --------------------------------------------------------------------------------------------------
# the work a pass cannot do without
# --------------------------------------------------------------------------------------------------
def _solve_flops(planes, h, w, s):
    """Two real 2-D transforms (LR forward, HR inverse) at 2.5 n log2 n each, and the spectral product."""
    n, N = h * w, h * w * s * s
    return planes * (2.5 * n * math.log2(max(2, n)) + 2.5 * N * math.log2(max(2, N)) + 4 * N)


def _block_flops(B, C, H, W, p):
    return 2 * B * H * W * 4 * (2 * C * C) + _solve_flops(2 * C * B, H + 2 * p, W + 2 * p, 1)


def work(case):
    c, kind = case, case["kind"]
    if kind == "dncnn":
        return {"bytes": 4 * (2 * c["B"] * c["H"] * c["W"] + 796353),
                "flops": 20 * _block_flops(c["B"], 64, c["H"], c["W"], 6) + 4 * 64 * c["B"] * c["H"] * c["W"]}
    if kind == "usrnet":
        H, W = c["H"] * c["s"], c["W"] * c["s"]
        return {"bytes": 4 * (3 * c["B"] * (c["H"] * c["W"] + H * W) + 950000),
                "flops": 35 * _block_flops(c["B"], 64, H, W, 2) + 5 * _solve_flops(64 * c["B"], H, W, 1)}
    B, C, H, W, k = c["B"], c["C"], c["H"], c["W"], c["k"]
    if kind == "block":
        return {"bytes": 4 * (2 * B * C * H * W + 8 * C * C + 2 * C * k * k),
                "flops": _block_flops(B, C, H, W, c["p"])}
    s = c["s"]
    n, N = B * C * H * W, B * C * H * W * s * s
    p = c.get("p", 0)
    f = _solve_flops(B * C, H + 2 * p, W + 2 * p, s)
    if kind == "op":
        return {"bytes": 4 * (n + 2 * N + C * k * k), "flops": f + 2.5 * N * math.log2(max(2, N // (B * C)))}
    if kind == "data":
        return {"bytes": 4 * (n + N + B * C * k * k), "flops": f}
    if kind == "train":  # x, grad_out read; out, grad_x written
        return {"bytes": 4 * (2 * n + 2 * N + 2 * C * k * k), "flops": 2 * f}
    return {"bytes": 4 * (n + N + C * k * k), "flops": f}


# --------------------------------------------------------------------------------------------------
# tolerances and 64-bit results
# --------------------------------------------------------------------------------------------------
def tolerance(case):
    # about four times the relative error seen against exact(): single layers 2e-7 to 9e-7 by size and lambda,
    # gradients up to 3e-7 (a bias gradient is a sum over whole planes), a block 1.1e-6, the 20-block denoiser
    # 1.4e-5, the 35-block unfolding network 4e-6 (its residual branches are scaled by small alphas)
    return {"rel": {"train": 1e-5, "block": 1e-5, "dncnn": 1e-4, "usrnet": 4e-5}.get(case["kind"], 4e-6)}


def _pad(x, p, mode):
    return x if p == 0 else F.pad(x, (p, p, p, p), mode=mode)


def _solve64(x, x0, psf, lam, s):
    """The closed-form solve in the form that does not divide by lambda:
    X = X0 + conj(K) (Y - mean(K X0)) / (mean |K|^2 + lambda), means over the s x s aliases of a bin."""
    B, C, h, w = x.shape
    H, W = h * s, w * s
    K = torch.zeros(psf.shape[0], C, H, W, dtype=x.dtype, device=x.device)
    kh, kw = psf.shape[-2:]
    i = (torch.arange(kh, device=x.device) - kh // 2) % H
    j = (torch.arange(kw, device=x.device) - kw // 2) % W
    K = K.index_put((torch.arange(psf.shape[0], device=x.device).view(-1, 1, 1, 1),
                     torch.arange(C, device=x.device).view(1, -1, 1, 1), i.view(1, 1, -1, 1), j.view(1, 1, 1, -1)),
                    psf, accumulate=True)
    K = torch.fft.fft2(K)

    def mean(a):
        return a.view(a.shape[0], C, s, h, s, w).mean((2, 4))

    X0 = torch.fft.fft2(x0)
    r = (torch.fft.fft2(x) - mean(K * X0)) / (mean(K.real ** 2 + K.imag ** 2) + lam)
    return torch.fft.ifft2(X0 + K.conj() * r.repeat(1, 1, s, s)).real


def _layer64(x, psf, bias, s, p, mode, eps):
    x = _pad(x, p, mode)
    x0 = x.repeat_interleave(s, 2).repeat_interleave(s, 3)
    y = _solve64(x, x0, psf, torch.sigmoid(bias - 9) + eps, s)
    return y[..., p * s:y.shape[2] - p * s, p * s:y.shape[3] - p * s]


def _ln64(x, w, b, eps):
    u = x.mean(1, keepdim=True)
    v = ((x - u) ** 2).mean(1, keepdim=True)
    return w.view(-1, 1, 1) * (x - u) / torch.sqrt(v + eps) + b.view(-1, 1, 1)


def _mix64(x, w, b):
    w = w.view(w.shape[0], -1)
    return torch.stack([(w @ t.flatten(1)).view(-1, *t.shape[1:]) for t in x]) + b.view(-1, 1, 1)


def _block64(x, d, pre, p, mode):
    q = {k[len(pre):]: v for k, v in d.items() if k.startswith(pre)}
    t = _ln64(x, q["conv1.0.weight"], q["conv1.0.bias"], 1e-5)
    t = F.gelu(_mix64(t, q["conv1.1.weight"], q["conv1.1.bias"]))
    t = F.gelu(_layer64(t, q["conv1.3.weight"], q["conv1.3.bias"], 1, p, mode, 1e-5))
    x = x + q.get("alpha1", 1.0) * _mix64(t, q["conv1.5.weight"], q["conv1.5.bias"])
    t = _ln64(x, q["conv2.0.weight"], q["conv2.0.bias"], 1e-5)
    t = F.gelu(_mix64(t, q["conv2.1.weight"], q["conv2.1.bias"]))
    return x + q.get("alpha2", 1.0) * _mix64(t, q["conv2.3.weight"], q["conv2.3.bias"])


def exact(case, seed):
    c, kind = case, case["kind"]
    st = prepare(case, seed)
    x = st["x"].detach().double()
    d = {k: v.detach().double() for k, v in st["net"].state_dict().items()} if "net" in st else {}
    if kind == "train":
        x.requires_grad_(True)
        w, b = d["weight"].requires_grad_(True), d["bias"].requires_grad_(True)
        out = _layer64(x, w, b, c["s"], c["p"], c["mode"], c["eps"])
        gx, gw, gb = torch.autograd.grad(out, (x, w, b), st["go"].double())
        return {"out": out.detach(), "gx": gx, "gw": gw, "gb": gb}
    with torch.no_grad():
        if kind == "layer":
            return _layer64(x, d["weight"], d["bias"], c["s"], c["p"], c["mode"], c["eps"])
        if kind == "op":
            return _solve64(x, st["x0"].double(), st["w"].double(), torch.sigmoid(st["b"].double() - 9) + c["eps"],
                            c["s"])
        if kind == "data":
            return _layer64(x, st["k"].double(), d["alpha"], c["s"], 0, "circular", 1e-3)
        if kind == "block":
            return _block64(x, d, "", c["p"], c["mode"])
        if kind == "dncnn":
            x = _mix64(x, d["m_head.0.weight"], d["m_head.0.bias"])
            for i in range(20):
                x = _block64(x, d, "m_body.%d." % i, 6, "circular")
            return _mix64(x, d["m_tail.0.weight"], d["m_tail.0.bias"])
        k = st["k"].double().flatten(1)
        for i in (1, 2, 3):
            k = k @ d["kernelnet.fc%d.weight" % i].t() + d["kernelnet.fc%d.bias" % i]
            k = F.gelu(k) if i < 3 else k
        k = k.view(c["B"], 16, c["k"], c["k"])
        x = _mix64(x, d["conv1.weight"], d["conv1.bias"])
        for i in range(5):
            psf = _mix64(k, d["convs.%d.weight" % i], d["convs.%d.bias" % i])
            # (B, 64, k, k) read as (B, 64, rows, columns) of the map
            x = _layer64(x, psf, d["d.alpha"], c["s"] if i == 0 else 1, 0, "circular", 1e-3)
            for j in range(7):
                x = _block64(x, d, "p.m_body.%d." % j, 2, "circular")
        return _mix64(x, d["conv2.weight"], d["conv2.bias"])
