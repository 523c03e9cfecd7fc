"""Transfer tables and scratch kept between calls, under what callers may do with them: views of one psf, several
streams, several host threads, captured graphs."""
import numpy as np
import pytest
import torch

from oracle import converse_oracle as O
from tests.conftest import seeded, softmax_psf

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
TOL = 1e-4  # largest difference at values near 1, as for the layer's other tests


def _case(seed, B=2, C=4, H=24, W=30, k=5):
    rng = seeded("gpu cache", seed)
    x = torch.from_numpy(rng.standard_normal((B, C, H, W)).astype(np.float32)).to(DEV)
    w = torch.from_numpy(softmax_psf(rng, C, k)).to(DEV)
    b = torch.from_numpy((0.2 * rng.standard_normal((1, C, 1, 1))).astype(np.float32)).to(DEV)
    return x, w, b


def _ref(x, w, b, s, p=0):
    a = [t.cpu().numpy() for t in (x, w, b)]
    return O.converse2d_module(a[0], a[1], a[2], s, p, "circular", 1e-5)


@pytest.mark.parametrize("entry", ["module", "op"])
def test_views_of_one_psf(entry):
    from conversenet_amd import functional as Fh

    x, w, b = _case("views")
    for v in (w, w.transpose(2, 3), w[:, :1].expand(w.shape), w):
        if entry == "module":
            got = Fh.converse2d_fused(x, v, b, 2, 0, "circular", 1e-5)
        else:
            x0 = x.repeat_interleave(2, 2).repeat_interleave(2, 3)
            got = Fh.converse2d_op(x, x0, v, b, 2, 1e-5)
        assert np.abs(got.cpu().numpy() - _ref(x, v, b, 2)).max() <= TOL
