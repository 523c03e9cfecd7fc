"""The channel-mixing kernels on pixel counts that are no multiple of 4, on buffers at any 4-byte alignment, and
on weights far from 1 (their split-fp16 parts are scaled per matrix), against the fp64 oracle.

Tolerance (relative 2-norm): the two operands and the dropped term of a split-fp16 product are off by 2^-22 each,
3 * 2^-22 = 7e-7 of it, with random signs (2^-25 of the pixel's largest activation for the smaller ones); GELU by
3.3e-7 absolute.  Through the three layers of a tail: 3 (7e-7 + 3.3e-7) = 3e-6 at most; fp32 rounding of the sums
adds 1e-7 each."""
import numpy as np
import pytest
import torch

from oracle import converse_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
TOL = 3e-6


def _t(a):
    """On the device, one float past a 16-byte boundary."""
    a = np.ascontiguousarray(a)
    buf = torch.empty(a.size + 1, device=DEV)
    v = buf[1:].view(a.shape)
    v.copy_(torch.from_numpy(a))
    return v


def _close(got, ref, what):
    got = got.cpu().numpy()
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= TOL, (what, err)


def _params(C, mid, seed, ws=1.0):
    r = np.random.default_rng(seed)
    f = lambda *s: r.standard_normal(s).astype(np.float32)  # noqa: E731
    return dict(lw=1 + 0.1 * f(C), lb=0.1 * f(C), w1=ws * f(mid, C, 1, 1) / np.float32(np.sqrt(C)), b1=f(mid),
                w2=f(C, mid, 1, 1) / np.float32(np.sqrt(mid) * ws), b2=f(C), w0=f(C, mid, 1, 1) / np.float32(np.sqrt(mid)),
                b0=f(C), a1=f(C), a2=f(C))


def _branch(y, p):
    return O.conv1x1(O.gelu(O.conv1x1(O.layernorm_cf(y, p["lw"], p["lb"], 1e-5), p["w1"], p["b1"])), p["w2"], p["b2"])


# pixel counts around one 16-pixel tile, one 256-pixel block and several blocks
SIZES = [(1, 1), (3, 5), (1, 17), (15, 17), (7, 37), (33, 65)]


@pytest.mark.parametrize("H,W", SIZES)
@pytest.mark.parametrize("head", [False, True])
def test_tail(H, W, head):
    from conversenet_amd import functional as Fh

    p = _params(64, 128, H * W)
    r = np.random.default_rng(W)
    t = r.standard_normal((2, 128, H, W)).astype(np.float32)
    x = r.standard_normal((2, 64, H, W)).astype(np.float32)
    s = lambda v: v[None, :, None, None]  # noqa: E731
    y1 = x + s(p["a1"]) * O.conv1x1(O.gelu(t), p["w0"], p["b0"])
    ref = y1 + s(p["a2"]) * _branch(y1, p)
    d = {k: _t(v) for k, v in p.items()}
    out = Fh.conv_ln_mlp_residual(_t(t), _t(x), d["w0"], d["b0"], d["lw"], d["lb"], 1e-5, d["w1"], d["b1"], d["w2"],
                                  d["b2"], d["a1"], d["a2"], t_act="gelu",
                                  head=(d["lw"], d["lb"], 1e-5, d["w1"], d["b1"]) if head else None)
    _close(out[0] if head else out, ref, "tail")
    if head:
        _close(out[1], O.gelu(O.conv1x1(O.layernorm_cf(ref, p["lw"], p["lb"], 1e-5), p["w1"], p["b1"])), "head")


@pytest.mark.parametrize("H,W", [(1, 1), (15, 17), (7, 37)])
@pytest.mark.parametrize("C,Cout", [(64, 64), (64, 16), (32, 32), (64, 32), (128, 64)])
def test_ln_conv_shapes(H, W, C, Cout):
    """The remaining LayerNorm shapes with split products, one pixel per lane."""
    from conversenet_amd import functional as Fh

    p = _params(C, Cout, 10 + C + Cout)
    x = np.random.default_rng(H + C).standard_normal((2, C, H, W)).astype(np.float32)
    d = {k: _t(v) for k, v in p.items()}
    got = Fh.conv1x1(_t(x), d["w1"], d["b1"], ln=(d["lw"], d["lb"], 1e-5))
    _close(got, O.conv1x1(O.layernorm_cf(x, p["lw"], p["lb"], 1e-5), p["w1"], p["b1"]), "ln conv")


@pytest.mark.parametrize("H,W", [(1, 1), (8, 9)])
@pytest.mark.parametrize("C,Cout", [(16, 64), (128, 128)])
def test_ln_conv_shapes_without_a_ragged_kernel(H, W, C, Cout):
    """fp32-product LayerNorm shapes: refused on ragged or misaligned input, as before."""
    from conversenet_amd import functional as Fh

    x, w, v = torch.zeros(1, C, H, W, device=DEV), torch.zeros(Cout, C, 1, 1, device=DEV), torch.ones(C, device=DEV)
    x = x if H * W % 4 else _t(x.cpu().numpy())
    with pytest.raises(RuntimeError, match="MFMA tile shape"):
        Fh.conv1x1(x, w, ln=(v, v, 1e-5))


@pytest.mark.parametrize("H,W", SIZES)
@pytest.mark.parametrize("C,mid", [(64, 128), (32, 64)])
def test_ln_conv_and_mlp(H, W, C, mid):
    from conversenet_amd import functional as Fh

    p = _params(C, mid, H + W)
    x = np.random.default_rng(H).standard_normal((2, C, H, W)).astype(np.float32)
    d = {k: _t(v) for k, v in p.items()}
    got = Fh.conv1x1(_t(x), d["w1"], d["b1"], act="gelu", ln=(d["lw"], d["lb"], 1e-5))
    _close(got, O.gelu(O.conv1x1(O.layernorm_cf(x, p["lw"], p["lb"], 1e-5), p["w1"], p["b1"])), "ln conv")
    got = Fh.ln_mlp_residual(_t(x), d["lw"], d["lb"], 1e-5, d["w1"], d["b1"], d["w2"], d["b2"], d["a2"])
    _close(got, x + p["a2"][None, :, None, None] * _branch(x, p), "mlp")


@pytest.mark.parametrize("ws", [1e-30, 1e-6, 300.0, 1e6])
def test_weight_scale(ws):
    """Weights whose fp16 parts would vanish or overflow without the per-matrix scale (1x1, no bias)."""
    from conversenet_amd import functional as Fh

    r = np.random.default_rng(3)
    x = r.standard_normal((1, 64, 9, 11)).astype(np.float32)
    w = (ws * r.standard_normal((128, 64, 1, 1)) / 8).astype(np.float32)
    _close(Fh.conv1x1(_t(x), _t(w)), O.conv1x1(x, w, np.zeros(128, np.float32)), ws)
    z = Fh.conv1x1(_t(x), _t(0 * w))
    assert not z.cpu().numpy().any()


SPLIT = [(64, 128, 9, 11), (128, 64, 5, 13), (64, 64, 8, 10), (32, 32, 6, 6)]  # ragged, and 16-byte vectors of pixels


def _conv_case(ci, co, H, W, seed):
    r = np.random.default_rng(seed)
    return r.standard_normal((2, ci, H, W)), (r.standard_normal((co, ci, 1, 1)) / np.sqrt(ci)).astype(np.float32)


def _conv(x, w):
    """On 16-byte aligned buffers (the vector forms)."""
    from conversenet_amd import functional as Fh

    return Fh.conv1x1(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV)).cpu().numpy()


@pytest.mark.parametrize("ci,co,H,W", SPLIT)
@pytest.mark.parametrize("sx,sw", [(1e-30, 1), (1e-6, 1), (1e-4, 1), (1e-2, 1), (0.3, 1), (1e5, 1), (1e20, 1e3),
                                   (1e36, 1e-3), (1e-3, 1e-30)])
def test_activation_scale(ci, co, H, W, sx, sw):
    """Activations (and weights with them) whose fp16 parts would vanish or overflow as they are."""
    x, w = _conv_case(ci, co, H, W, 7)
    x, w = (sx * x).astype(np.float32), np.float32(sw) * w
    ref = np.einsum("oc,bchw->bohw", w[:, :, 0, 0].astype(np.float64), x.astype(np.float64))
    got = _conv(x, w)
    assert np.isfinite(got).all()
    assert np.linalg.norm((got - ref) / sx / sw) <= TOL * np.linalg.norm(ref / sx / sw)


@pytest.mark.parametrize("ci,co,H,W", SPLIT)
def test_large_activation_in_a_late_channel(ci, co, H, W):
    """Pixels that fit by their first 32 channels, with one above fp16's end in the last: the products start over."""
    x, w = _conv_case(ci, co, H, W, 11)
    x = x.astype(np.float32)
    x[0, -1, 1, 2], x[1, -1, 0, 0] = 3e5, -1e30
    ref = np.einsum("oc,bchw->bohw", w[:, :, 0, 0].astype(np.float64), x.astype(np.float64))
    assert (np.linalg.norm(_conv(x, w) - ref, axis=1) <= TOL * np.linalg.norm(ref, axis=1)).all()


@pytest.mark.parametrize("ci,co,H,W", SPLIT)
def test_pixels_and_rows_of_different_size(ci, co, H, W):
    """Pixels 1e-8 to 1e8, each against its own size (they are scaled one by one); an infinity stays in its pixel, and
    is one there; output rows 1e-2.5 to 1e2.5 (a matrix has one scale: a row is exact to 2^-22 from 2^-17 of the largest
    entry on)."""
    r = np.random.default_rng(8)
    x, w = _conv_case(ci, co, H, W, 9)
    x = (x * 10.0 ** r.uniform(-8, 8, (2, 1, H, W))).astype(np.float32)
    x[0, :, 0, 0] = 0
    ref = np.einsum("oc,bchw->bohw", w[:, :, 0, 0].astype(np.float64), x.astype(np.float64))
    got = _conv(x, w)
    assert not got[0, :, 0, 0].any()
    assert (np.linalg.norm(got - ref, axis=1) <= TOL * np.linalg.norm(ref, axis=1)).all()
    x[1, 3, 2, 1] = np.inf
    got2 = _conv(x, w)
    assert (got2[1, :, 2, 1] == np.sign(w[:, 3, 0, 0]) * np.inf).all()
    got2[1, :, 2, 1], ref[1, :, 2, 1] = 0, 0
    assert (np.linalg.norm(got2 - ref, axis=1) <= TOL * np.linalg.norm(ref, axis=1)).all()
    x = r.standard_normal((2, ci, H, W)).astype(np.float32)
    w = (w * 10.0 ** r.uniform(-2.5, 2.5, (co, 1, 1, 1))).astype(np.float32)
    ref = np.einsum("oc,bchw->bohw", w[:, :, 0, 0].astype(np.float64), x.astype(np.float64))
    size = lambda a: np.sqrt((a ** 2).sum((0, 2, 3)))  # noqa: E731
    assert (size(_conv(x, w) - ref) <= TOL * size(ref)).all()


@pytest.mark.parametrize("mode,k,pad", [("circular", 7, 6), ("replicate", 5, 4)])
def test_block_and_chain_on_odd_images(mode, k, pad):
    """A block and a chain of blocks on 45 x 41 pixels (padded planes 57 x 53 and 53 x 49)."""
    from conversenet_amd.util_converse import ConverseBlock, run_blocks

    torch.manual_seed(1)
    blks = [ConverseBlock(64, 64, kernel_size=k, padding=pad, padding_mode=mode).to(DEV).eval() for _ in range(3)]
    x = np.random.default_rng(2).standard_normal((2, 64, 45, 41)).astype(np.float32)
    ref = x
    for b in blks:
        sd = {n: v.detach().cpu().numpy() for n, v in b.state_dict().items()}
        ref = O.converse_block(ref, sd, "", k, 1, pad, mode, 1e-5, False)
    with torch.no_grad():
        _close(run_blocks(blks, _t(x)), ref, "chain")
        y = _t(x)
        for b in blks:
            y = b(y)
    _close(y, ref, "blocks")


def _every_other(t):
    """The same values with gaps between them: a wrapper copies it to pass it on."""
    return torch.stack([t, torch.full_like(t, 9.0)], -1)[..., 0] if t is not None else None


def test_strided_parameters():
    """Parameters that a wrapper has to copy: every copy keeps its memory until the kernels are enqueued."""
    from conversenet_amd import functional as Fh

    p = {k: torch.from_numpy(v).to(DEV) for k, v in _params(64, 128, 5).items()}
    r = np.random.default_rng(6)
    x, t = (torch.from_numpy(r.standard_normal((1, c, 9, 13)).astype(np.float32)).to(DEV) for c in (64, 128))

    def calls(d):
        ln = (d["lw"], d["lb"], 1e-5)
        yield Fh.layernorm_cf(x, *ln)
        yield Fh.conv1x1(t, d["w0"], d["b0"], residual=x, res_scale=d["a1"])
        yield Fh.conv1x1(x, d["w1"], d["b1"], ln=ln)
        yield Fh.ln_mlp_residual(x, *ln, d["w1"], d["b1"], d["w2"], d["b2"], d["a2"])
        yield from Fh.conv_ln_mlp_residual(t, x, d["w0"], d["b0"], *ln, d["w1"], d["b1"], d["w2"], d["b2"], d["a1"],
                                           d["a2"], head=(*ln, d["w1"], d["b1"]))

    for n, (a, b) in enumerate(zip(calls(p), calls({k: _every_other(v) for k, v in p.items()}))):
        assert torch.equal(a, b), n
