"""The in-place prime-factor row and column passes (csrc/fft_lines.h) against the fp64 oracle: every length
up to 1024, so every radix, every Cooley-Tukey part and every dense prime, in rows and in columns.

Tolerance (relative 2-norm): a call makes four transforms, each of at most 5 rounded operations per pass and
element, 3 passes; at 6e-8 per rounding and independent errors that is 4 sqrt(15) 6e-8 = 9e-7.  A dense prime adds
chunked sums of up to 512 terms, sqrt((32 + 512 / 32) / 6) roundings, 4 * 2.8 * 6e-8 = 7e-7.  Gate: 3e-6, above the
sum of both."""
import numpy as np
import pytest
import torch

from oracle import converse_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
TOL = 3e-6


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _inputs(B, C, H, W, k, seed, pb=1):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((B, C, H, W)).astype(np.float32)
    w = rng.random((pb, C, k, k))
    w = (w / w.sum(axis=(2, 3), keepdims=True)).astype(np.float32)
    b = (0.3 * rng.standard_normal((1, C, 1, 1))).astype(np.float32)
    return x, w, b


def _check(x, w, b, s, p, mode, what):
    from conversenet_amd import functional as Fh

    ref = O.converse2d_module(x, w, b, s, p, mode, 1e-5)
    got = Fh.converse2d_fused(_t(x), _t(w), _t(b).reshape(-1), s, p, mode, 1e-5, cache=False).cpu().numpy()
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= TOL, (what, err)


@pytest.mark.parametrize("first", range(1, 1025, 128))
def test_every_length(first):
    """Rows of L samples (5 rows: an odd count leaves half a pair) and columns of L samples."""
    for L in range(first, first + 128):
        for H, W in ((5, L), (L, 3)):
            x, w, b = _inputs(1, 2, H, W, 1 if min(H, W) < 3 else 3, L)
            _check(x, w, b, 1, 0, "circular", (H, W))


@pytest.mark.parametrize("part", range(4))
def test_lengths_with_a_kernel_for_few_blocks(part):
    """Lengths whose rows or columns run on another kernel at two planes, on enough planes for this one, and on the
    largest number that keeps the other."""
    from conversenet_amd import _lib

    lib = _lib.load()

    def cols(P, L):
        return lib.cvn_converse2d_column_pass(_lib.CALL_MODULE, 1, P, L, 3, 1, 1, 0)

    def rows(P, L):
        return lib.cvn_converse2d_row_pass(P, 1, L)

    seen = [0, 0]
    for L in range(1 + part, 1025, 4):
        for n, (kernel, H, W) in enumerate(((rows, 1, L), (cols, L, 3))):
            if kernel(2, L) == _lib.COLS_LINES:
                continue
            lo, hi = 2, 4096  # the last count on the other kernel, the first on this one
            while hi - lo > 1:
                mid = (lo + hi) // 2
                lo, hi = (mid, hi) if kernel(mid, L) == _lib.COLS_SINGLE else (lo, mid)
            assert kernel(hi, L) == _lib.COLS_LINES
            seen[n] += 1
            for P in (lo, hi):
                x, w, b = _inputs(1, P, H, W, 1, L)
                _check(x, w, b, 1, 0, "circular", (P, H, W))
    assert min(seen) >= 1


# (B, C, H, W, k, s, p, mode, psf batch): blocks that straddle planes and channels, odd rows and crops, a
# mirrored LR column at s > 1, dense primes (37, 61, 127) and staged parts (49, 64, 81, 343) in both directions
CASES = [
    (3, 5, 31, 29, 3, 1, 4, "circular", 1),     # 39 x 37
    (2, 3, 33, 57, 5, 1, 2, "reflect", 2),      # 37 x 61
    (2, 3, 55, 123, 7, 1, 3, "replicate", 1),   # 61 x 129
    (1, 2, 115, 331, 7, 1, 6, "constant", 1),   # 127 x 343
    (2, 7, 20, 23, 2, 2, 2, "replicate", 1),    # 48 x 54
    (1, 3, 15, 25, 3, 3, 1, "circular", 1),     # 51 x 81
    (2, 2, 12, 33, 5, 4, 2, "reflect", 2),      # 64 x 148
    (1, 2, 60, 41, 3, 2, 1, "constant", 1),     # 124 x 86
    (2, 2, 130, 91, 3, 5, 2, "circular", 1),    # 670 x 475: scale above 4
    (1, 1, 250, 1, 3, 4, 2, "replicate", 1),    # 1016 x 20
    (1, 2, 508, 3, 3, 2, 2, "circular", 1),     # 1024 x 14: the largest column buffer, most LR rows per thread
    (2, 3, 3, 4, 3, 3, 0, "circular", 1),       # 9 x 12: LR rows fewer than a wave's items
    (3, 2, 41, 6, 2, 2, 1, "reflect", 1),       # 86 x 16: 43 LR rows, items in an uneven last round
]


@pytest.mark.parametrize("B,C,H,W,k,s,p,mode,pb", CASES)
def test_shapes_modes_scales(B, C, H, W, k, s, p, mode, pb):
    x, w, b = _inputs(B, C, H, W, k, 7 * H + W, pb)
    _check(x, w, b, s, p, mode, (H, W, s, p))


# (B, C, h, w, k, s, lines): even and odd w (self-mirrored classes 0 and w / 2, the middle member of an odd scale),
# dense and staged lengths, each with classes enough for the lines pass; too few of them, and a length (500 rows at
# s = 2) whose members exceed LDS, which stay on the class-per-block pass
OP_CASES = [
    (2, 40, 21, 37, 3, 1, True),
    (3, 33, 15, 26, 3, 2, True),
    (2, 54, 49, 17, 5, 3, True),
    (2, 40, 9, 24, 3, 3, True),
    (2, 92, 10, 12, 7, 4, True),
    (1, 120, 7, 21, 3, 4, True),
    (1, 97, 37, 31, 2, 2, True),
    (2, 30, 49, 17, 5, 3, False),
    (2, 80, 10, 12, 7, 4, False),
    (2, 14, 250, 44, 3, 2, False),
]


@pytest.mark.parametrize("B,C,h,w,k,s,lines", OP_CASES)
def test_operator_arbitrary_x0(B, C, h, w, k, s, lines):
    from conversenet_amd import _lib
    from conversenet_amd import functional as Fh

    assert _lib.load().cvn_converse2d_column_pass(_lib.CALL_OP, B, C, h, w, 1, s, 0) == int(lines)
    x, psf, b = _inputs(B, C, h, w, k, h * w)
    x0 = np.random.default_rng(w).standard_normal((B, C, h * s, w * s)).astype(np.float32)
    ref = O.converse2d_op_stable(x, x0, psf, b, s, 1e-5)
    got = Fh.converse2d_op(_t(x), _t(x0), _t(psf), _t(b), s, 1e-5, cache=False).cpu().numpy()
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= TOL, err


# (B, C, H, W, k, s, p, mode, psf batch, lines): several planes per psf and blocks that straddle psf groups
BWD_CASES = [
    (3, 5, 31, 29, 3, 1, 4, "circular", 1, True),  # 39 x 37
    (2, 3, 33, 57, 5, 1, 2, "reflect", 2, True),  # 37 x 61
    (4, 3, 94, 43, 3, 1, 3, "replicate", 1, True),  # 100 x 49
    (3, 4, 15, 26, 3, 2, 1, "constant", 1, True),  # 34 x 56
    (2, 3, 17, 13, 5, 3, 2, "circular", 2, False),  # 63 x 51: few blocks, one plane per psf
    (2, 135, 5, 20, 5, 3, 2, "circular", 2, True),  # 27 x 72
    (3, 2, 10, 21, 2, 4, 1, "reflect", 1, False),  # 48 x 92
    (1, 5, 16, 20, 3, 2, 0, "circular", 1, True),  # 32 x 40: one plane per psf, the lines pass
    (2, 60, 14, 110, 3, 2, 0, "circular", 1, True),  # 28 x 220: blocks for most of the chip, the lines pass
    (8, 3, 24, 10, 3, 1, 0, "circular", 1, False),  # 24 x 10: few blocks, a column class or more per block
    (4, 2, 100, 9, 3, 3, 1, "replicate", 1, True),  # 306 x 33 (17 a factor): the lines pass at few blocks
    (3, 3, 70, 9, 3, 3, 0, "constant", 1, False),  # 210 x 27: few blocks of long columns
]


@pytest.mark.parametrize("B,C,H,W,k,s,p,mode,pb,lines", BWD_CASES)
@pytest.mark.parametrize("weights", [True, False])
def test_backward(B, C, H, W, k, s, p, mode, pb, lines, weights):
    from conversenet_amd import _lib
    from conversenet_amd import functional as Fh

    assert _lib.load().cvn_converse2d_column_pass(_lib.CALL_BWD, B, C, H, W, pb, s, p) == int(lines)
    x, w, b = _inputs(B, C, H, W, k, H + W, pb)
    go = np.random.default_rng(W).standard_normal((B, C, H * s, W * s)).astype(np.float32)
    ref = O.converse2d_module_backward(x, w, b, go, s, p, mode, 1e-5)
    got = Fh.converse2d_backward(_t(go), _t(x), _t(w), _t(b), s, p, mode, 1e-5, True, weights, weights)
    for g, r in zip(got[:3 if weights else 1], ref):
        r = np.asarray(r).reshape(g.shape)
        # the weight gradients are sums over all bins in fp64 of products that are right to TOL
        assert np.linalg.norm(g.cpu().numpy() - r) / np.linalg.norm(r) <= TOL


def test_misaligned_scratch_and_infinite_plane():
    """Spectra scratch at 8 bytes past a 16-byte boundary (no 16-byte accesses), and a plane of infinities and
    NaN that shares its blocks with finite planes, which it must not touch."""
    from conversenet_amd import _lib
    from conversenet_amd import functional as Fh

    x, w, b = _inputs(3, 2, 34, 44, 3, 5)
    x[1, 0] = np.nan
    x[1, 1, 3, 4] = np.inf
    ref = O.converse2d_module(np.where(np.isfinite(x), x, 0), w, b, 1, 1, "circular", 1e-5)
    xt, wt, bt = _t(x), _t(w), _t(b).reshape(-1)
    got = Fh.converse2d_fused(xt, wt, bt, 1, 1, "circular", 1e-5, cache=False).cpu().numpy()
    lib = _lib.load()
    geo = (3, 2, 34, 44, 1, 3, 3, 1, 1)
    route, mode = lib.cvn_converse2d_route(*geo), _lib.PAD_MODES["circular"]
    tb, sb = lib.cvn_converse2d_table_bytes(*geo, route), lib.cvn_converse2d_scratch_bytes(*geo, route)
    table = torch.empty(tb, dtype=torch.uint8, device=DEV)
    scratch = torch.empty(sb + 8, dtype=torch.uint8, device=DEV)
    out = torch.empty(3, 2, 34, 44, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    assert lib.cvn_converse2d_table_f32(wt.data_ptr(), 1, 3, 3, bt.data_ptr(), 1e-5, 3, 2, 34, 44, 1, 1, route,
                                        table.data_ptr(), tb, st) == 0
    assert lib.cvn_converse2d_apply_f32(xt.data_ptr(), 3, 2, 34, 44, 1, 3, 3, 1, 1, mode, 0, route, table.data_ptr(), tb,
                                        scratch.data_ptr() + 8, sb, out.data_ptr(), st) == 0
    for y in (got, out.cpu().numpy()):
        for i in (0, 2):
            assert np.linalg.norm(y[i] - ref[i]) / np.linalg.norm(ref[i]) <= TOL
        assert np.isnan(y[1]).all()
