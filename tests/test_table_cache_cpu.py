"""Host-side transfer-table cache policy (conversenet_amd.functional.TableCache, cacheable) and the
module's routing of unsupported geometries, on CPU tensors (no device needed)."""
import torch

from conversenet_amd import functional as Fh


def _key(w, b, geo=(1,), route=1):
    return Fh._cache_key("module", w, b, 1e-5, geo, route, torch.device("cpu"))


def test_in_place_update_replaces_entry_instead_of_adding():
    c = Fh.TableCache()
    w, b = torch.ones(1, 4, 3, 3), torch.zeros(1, 4, 1, 1)
    c.put(_key(w, b), torch.empty(100, dtype=torch.uint8), (w, b))
    assert c.get(_key(w, b)) is not None
    for _ in range(5):  # optimizer-style in-place steps
        w.mul_(0.5)
        assert c.get(_key(w, b)) is None
        c.put(_key(w, b), torch.empty(100, dtype=torch.uint8), (w, b))
    assert len(c.entries) == 1 and c.bytes == 100


def test_route_and_geometry_are_part_of_the_key():
    c = Fh.TableCache()
    w, b = torch.ones(1, 4, 3, 3), torch.zeros(1, 4, 1, 1)
    c.put(_key(w, b, route=1), torch.empty(10, dtype=torch.uint8), (w, b))
    assert c.get(_key(w, b, route=3)) is None
    assert c.get(_key(w, b, geo=(2,))) is None
    c.put(_key(w, b, route=3), torch.empty(20, dtype=torch.uint8), (w, b))
    assert len(c.entries) == 2 and c.bytes == 30


def test_views_of_one_address_have_tables_of_their_own():
    """A transposed square psf, and rows of one psf expanded, start at the address of the tensor they view."""
    c = Fh.TableCache()
    w, b = torch.rand(1, 4, 3, 3), torch.zeros(1, 4, 1, 1)
    views = [(w, b), (w.transpose(2, 3), b), (w[:, :1].expand(1, 4, 3, 3), b), (w, b[:, :1].expand(1, 4, 1, 1))]
    assert len({(v.data_ptr(), v._version, u.data_ptr(), u._version) for v, u in views}) == 1
    for n, (v, u) in enumerate(views):
        assert c.get(_key(v, u)) is None, n
        c.put(_key(v, u), torch.full((10,), n, dtype=torch.uint8), (v, u))
    for n, (v, u) in enumerate(views):
        assert int(c.get(_key(v, u))[0]) == n


def test_lru_bounds():
    c = Fh.TableCache(max_entries=3, max_bytes=250)
    ts = [(torch.ones(1, 1, 1, 1), torch.zeros(1, 1, 1, 1)) for _ in range(5)]
    for w, b in ts:
        c.put(_key(w, b), torch.empty(100, dtype=torch.uint8), (w, b))
    assert len(c.entries) == 2 and c.bytes == 200
    assert c.get(_key(*ts[-1])) is not None and c.get(_key(*ts[0])) is None
    c.clear()
    assert c.bytes == 0 and not c.entries and not c.latest


def test_entries_keep_the_memory_of_reassigned_parameters():
    """p.data = t (Module.to, weight swaps) leaves the version as it is: an address that returned to the
    allocator could come back with other values under the same key."""
    c = Fh.TableCache()
    w = torch.nn.Parameter(torch.ones(1, 4, 3, 3))
    b = torch.nn.Parameter(torch.zeros(1, 4, 1, 1))
    old = [(t.data_ptr(), t.detach().clone()) for t in (w, b)]
    k = _key(w, b)
    c.put(k, torch.empty(100, dtype=torch.uint8), (w, b))
    for t in (w, b):
        t.data = torch.full_like(t, 2.0)
    held = {t.data_ptr(): t for t in c.entries[k][1]}
    assert all(p in held and torch.equal(held[p], v) for p, v in old)
    assert c.get(_key(w, b)) is None


def test_psf_stack_follows_the_convolutions(monkeypatch):
    """The weights that ConverseUSRNet stacks: reassigned through .data (the version stays, and the old memory may
    come back under the same address with other values), updated in place, and made in inference mode."""
    from conversenet_amd import converse_usrnet as M

    seen = []  # the stacked weights and biases that each forward used
    monkeypatch.setattr(M, "_hip_eligible", lambda *ts: True)
    monkeypatch.setattr(Fh, "conv1x1", lambda k, w, b: (seen.append((w.clone(), b.clone())),
                                                        torch.nn.functional.conv2d(k, w, b))[1])
    monkeypatch.setattr(Fh, "table_cache", Fh.TableCache())
    monkeypatch.setattr(Fh, "_stream", lambda dev: None)

    class Net:
        pass

    def check(net):
        k = torch.rand(2, 16, 3, 3)
        with torch.no_grad():
            maps = M._psf_maps(net, k, 2, 3, 3)
            for c, got in zip(net.convs, maps):
                assert torch.equal(got, c(k).view(2, 64, 3, 3)) or torch.allclose(got, c(k).view(2, 64, 3, 3), atol=1e-6)
        w, b = seen[-1]
        assert torch.equal(w, torch.cat([c.weight for c in net.convs]))
        assert torch.equal(b, torch.cat([c.bias for c in net.convs]))

    net = Net()
    net.convs = [torch.nn.Conv2d(16, 64, 1) for _ in range(3)]
    check(net)
    ps = [t for c in net.convs for t in (c.weight, c.bias)]
    old = [(t.data_ptr(), t.detach().clone()) for t in ps]
    for t in ps:
        t.data = torch.rand_like(t)
    held = {t.data_ptr(): t for _, refs in Fh.table_cache.entries.values() for t in refs}
    assert all(p in held and torch.equal(held[p], v) for p, v in old)
    check(net)
    with torch.no_grad():
        net.convs[1].weight.mul_(2)
    check(net)
    with torch.inference_mode():
        net.convs = [torch.nn.Conv2d(16, 64, 1) for _ in range(3)]
        check(net)


def _fake_streams(monkeypatch):
    """Tables' stream ordering written down instead of enqueued; state["capturing"]: the streams that record a graph."""
    log, state = [], {"capturing": set()}

    class Made:
        def __init__(self, dev, stream):
            self.made_on, self.streams = stream, {stream}
            log.append(("made", stream))

        def join(self, table, stream):
            if self.made_on in state["capturing"]:
                return False
            self.streams.add(stream)
            log.append(("wait and hold", stream))
            return True

        def finish(self):
            log.append(("host wait",))

    monkeypatch.setattr(Fh, "_Made", Made)
    monkeypatch.setattr(Fh, "_capturing", lambda s: s in state["capturing"])
    return log, state


def test_hits_wait_for_the_stream_that_made_the_table(monkeypatch):
    log, state = _fake_streams(monkeypatch)
    c = Fh.TableCache()
    w, b = torch.ones(1, 4, 3, 3), torch.zeros(1, 4, 1, 1)
    c.put(_key(w, b), torch.empty(8, dtype=torch.uint8), (w, b), 7)
    assert c.get(_key(w, b), 7) is not None and log == [("made", 7)]
    assert c.get(_key(w, b), 9) is not None and log[1:] == [("wait and hold", 9)]
    state["capturing"] = {7}  # no wait for a stream that records a graph: the call makes its own table
    assert c.get(_key(w, b), 8) is None
    state["capturing"] = set()
    assert c.get(_key(w, b), 8) is not None


def test_tables_and_recorded_graphs(monkeypatch):
    """A table made while its stream records a graph is not kept; one made before is waited for, and stays while a
    graph may read it: until the psf's memory is released."""
    log, state = _fake_streams(monkeypatch)
    c = Fh.TableCache(max_entries=2)
    state["capturing"] = {5}
    w, b = torch.ones(1, 4, 3, 3), torch.zeros(1, 4, 1, 1)
    c.put(_key(w, b), torch.empty(8, dtype=torch.uint8), (w, b), 5)
    assert not c.entries and c.get(_key(w, b), 0) is None
    c.put(_key(w, b), torch.empty(8, dtype=torch.uint8), (w, b), 0)
    t = c.get(_key(w, b), 5)
    assert t is not None and ("host wait",) in log and len(c.recorded) == 1
    w.add_(1)
    c.put(_key(w, b), torch.empty(8, dtype=torch.uint8), (w, b), 0)
    c.clear()
    assert any(r is t for _, r in c.recorded)  # replaced, then cleared: the graph still reads it
    others = [(torch.ones(1, 1, 3, 3), b) for _ in range(2)]
    for n, (v, u) in enumerate(others):
        c.put(_key(v, u), torch.empty(8, dtype=torch.uint8), (v, u), 0)
        assert (c.get(_key(v, u), 5) is not None) == (n == 0)  # at most max_entries: then a graph makes its own
    del w
    assert c.get(_key(*others[1]), 5) is not None and not any(r is t for _, r in c.recorded)


def test_cacheable_rules():
    w = torch.nn.Parameter(torch.ones(1, 4, 3, 3))
    b = torch.nn.Parameter(torch.zeros(1, 4, 1, 1))
    assert not Fh.cacheable(w, b)  # autograd tracks them: training
    with torch.no_grad():
        assert Fh.cacheable(w, b)
    with torch.inference_mode():
        assert Fh.cacheable(w, b)  # parameters created outside inference mode keep a version counter
        k = torch.ones(1, 4, 3, 3)  # an activation made in inference mode (ConvReverseDataNet's psf)
        assert k.is_inference() and not Fh.cacheable(k, b)


def test_unsupported_geometries_are_routed_to_the_composition():
    w = torch.ones(1, 3, 3, 3) / 9
    assert Fh.supported(torch.empty(1, 3, 64, 64), w, 1, 1)
    assert not Fh.supported(torch.empty(1, 3, 5000, 8), w, 1, 1)
    assert not Fh.supported(torch.empty(1, 3, 8, 8), w, 5, 1, grad_weight=True)
    assert Fh.supported(torch.empty(1, 3, 8, 8), w, 5, 1, grad_x=True)
    assert Fh.supported(None, w, 1, 1, shape=(1, 3, 64, 64))


def test_concurrent_callers_keep_the_cache_consistent():
    """The op may be called from any host thread (the reference's cache is mutex-guarded,
    converse2d.cpp:56,70,90): eight threads hitting, filling and invalidating (in-place updates) one
    cache leave its byte count, entry bound and latest-version map consistent and raise nothing."""
    import random
    import threading

    c = Fh.TableCache(max_entries=16, max_bytes=1 << 30)
    params = [(torch.ones(1, 1, 1, 1), torch.zeros(1, 1, 1, 1)) for _ in range(40)]
    errors = []
    start = threading.Barrier(8)

    def worker(seed):
        rng = random.Random(seed)
        start.wait()
        try:
            for _ in range(3000):
                w, b = params[rng.randrange(len(params))]
                k = _key(w, b)
                if c.get(k) is None:
                    c.put(k, torch.empty(rng.choice((10, 20, 30)), dtype=torch.uint8), (w, b))
                if rng.random() < 0.05:
                    w.add_(0)  # an in-place update: bumps the version counter
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[:3]
    assert len(c.entries) <= 16
    assert c.bytes == sum(t.numel() for t, _ in c.entries.values())
    assert all(c.latest[c._stem(k)] == k for k in c.entries)


def test_scratch_belongs_to_one_call_at_a_time(monkeypatch):
    """Two threads on one stream: the second call's kernels follow the first's; a graph's call has its own buffer."""
    import threading

    dev = torch.device("cpu")
    monkeypatch.setattr(Fh, "_capturing", lambda s: s == 5)
    inside, go_on, order = threading.Event(), threading.Event(), []

    def first():
        ws = Fh._scratch(dev, 0)
        with ws.lock:
            order.append(("first in", ws.ptr(1000)))
            inside.set()
            go_on.wait(10)
            order.append(("first out", ws.ptr(500)))

    def second():
        inside.wait(10)
        ws = Fh._scratch(dev, 0)
        with ws.lock:
            order.append(("second in", ws.ptr(1000)))

    ts = [threading.Thread(target=f) for f in (first, second)]
    for t in ts:
        t.start()
    inside.wait(10)
    ts[1].join(0.2)
    assert ts[1].is_alive()  # waits for the first
    assert Fh._scratch(dev, 9).lock.acquire(blocking=False)  # another stream does not
    go_on.set()
    for t in ts:
        t.join(10)
    assert [n for n, _ in order] == ["first in", "first out", "second in"] and len({p for _, p in order}) == 1
    g, g2 = Fh._scratch(dev, 5), Fh._scratch(dev, 5)
    assert g is not g2 and g.ptr(10) != g2.ptr(10)
    assert (None, 5) not in Fh._ws_cache
    Fh.release_workspace()
    assert not Fh._ws_cache
