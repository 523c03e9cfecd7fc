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


def test_table_made_on_another_stream():
    """A hit waits for a table that is still being made on another stream (delayed there by a spinning kernel)."""
    from conversenet_amd import functional as Fh

    x, w, b = _case("streams", C=64, H=40, W=40)
    refs = [_ref(x, w, b, 2), _ref(x, w, b, 1)]
    a, s = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        torch.cuda._sleep(20_000_000)
        Fh.converse2d_fused(x, w, b, 2, 0, "circular", 1e-5)
        Fh.converse2d_fused(x, w, b, 1, 0, "circular", 1e-5)
    with torch.cuda.stream(s):
        hits = Fh.table_cache.hits
        got = [Fh.converse2d_fused(x, w, b, n, 0, "circular", 1e-5) for n in (2, 1)]
        assert Fh.table_cache.hits == hits + 2
    torch.cuda.synchronize()
    for g, r in zip(got, refs):
        assert np.abs(g.cpu().numpy() - r).max() <= TOL


@pytest.mark.parametrize("warm", [False, True])
def test_recorded_graph(warm):
    """A recorded call without its table makes one in the graph, for itself alone; with one from before, the table
    outlives the cache's entry.  Replays between other work, each against the eager result."""
    from conversenet_amd import functional as Fh

    x, w, b = _case(("graph", warm), C=16, H=36, W=28)
    ref = _ref(x, w, b, 2)
    if warm:
        Fh.converse2d_fused(x, w, b, 2, 0, "circular", 1e-5)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = Fh.converse2d_fused(x, w, b, 2, 0, "circular", 1e-5)
    misses = Fh.table_cache.misses
    got = Fh.converse2d_fused(x, w, b, 2, 0, "circular", 1e-5)  # eager, the graph has not run yet
    assert Fh.table_cache.misses == misses + (not warm)
    assert np.abs(got.cpu().numpy() - ref).max() <= TOL
    torch.ops.converse2d.clear_cache()
    for n in range(3):
        junk = [torch.full((1 << 18,), float("nan"), device=DEV) for _ in range(40)]  # takes over what was released
        x2 = x * (n + 1)
        eager = Fh.converse2d_fused(x2, w, b, 2, 0, "circular", 1e-5)
        keep = x.clone()
        x.copy_(x2)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), n
        x.copy_(keep)
        del junk


def test_two_threads_on_one_stream():
    """Calls of two threads on the default stream, on the multi-pass route: each thread's results are its own."""
    import threading

    from conversenet_amd import functional as Fh

    cases = [_case(("threads", n), C=8, H=40 + 4 * n, W=36) for n in range(2)]
    want = [Fh.converse2d_fused(*c, 2, 0, "circular", 1e-5) for c in cases]
    wrong, start = [], threading.Barrier(2)

    def work(n):
        start.wait()
        for i in range(50):
            got = Fh.converse2d_fused(*cases[n], 2, 0, "circular", 1e-5)
            if not torch.equal(got, want[n]):
                wrong.append((n, i))

    ts = [threading.Thread(target=work, args=(n,)) for n in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong, wrong[:5]


def test_graph_keeps_its_scratch():
    """A graph recorded on the stream of the calls before it, which grow that stream's scratch afterwards."""
    from conversenet_amd import functional as Fh

    x, w, b = _case("graph scratch", C=8, H=36, W=36)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        want = Fh.converse2d_fused(x, w, b, 2, 0, "circular", 1e-5)
    with torch.cuda.graph(g, stream=s):
        out = Fh.converse2d_fused(x, w, b, 2, 0, "circular", 1e-5)
    big = torch.randn(4, 8, 96, 96, device=DEV)
    for n in range(3):
        with torch.cuda.stream(s):
            Fh.converse2d_fused(big[: n + 2], w, b, 2, 0, "circular", 1e-5)
            canary = [torch.zeros(1 << 16, device=DEV) for _ in range(20)]
        s.synchronize()
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and not any(c.any() for c in canary)
