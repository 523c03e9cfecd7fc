"""Tensor-level wrappers over the HIP C ABI (fp32, HIP device tensors only, forward only).

Each wrapper validates shapes the way the reference does (TORCH_CHECK -> RuntimeError,
Converse2D/torch_converse2d/converse2d.cpp:167-172), makes inputs contiguous like the reference op
(:174-177), allocates outputs and workspace through torch's caching allocator and enqueues the
kernels on torch's current stream.  No CPU fallback exists here: a missing library raises.
"""
from __future__ import annotations

import ctypes
import os
import threading

import torch
from torch.multiprocessing.reductions import StorageWeakRef

from . import _lib, composite

# The op is callable from any host thread (the reference guards its OTF cache with a mutex,
# converse2d.cpp:56,70,90): the workspace map, the plan memo and the table cache each take a lock
# around their dict updates.  Table builds run outside the locks, launches that use a stream's scratch under
# that scratch's own lock.
_ws_cache: dict = {}
_ws_lock = threading.Lock()


def _stream(dev):
    """The current stream's handle.  (torch.cuda.current_stream builds a Stream object around it: 2 us, as much
    host time as a kernel launch.)"""
    return torch._C._cuda_getCurrentRawStream(dev.index)


def _need_hip(*ts):
    for t in ts:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError("conversenet_amd HIP path needs tensors on a HIP device")
        if t.dtype != torch.float32:
            raise RuntimeError("conversenet_amd HIP path computes in float32")


class _Scratch:
    """A uint8 buffer that grows; `lock` is held while a call that uses it enqueues its kernels."""

    __slots__ = ("dev", "lock", "buf")

    def __init__(self, dev):
        self.dev, self.lock, self.buf = dev, threading.Lock(), None

    def ptr(self, nbytes):
        if nbytes == 0:
            return None
        if self.buf is None or self.buf.numel() < nbytes:
            self.buf = torch.empty(nbytes, dtype=torch.uint8, device=self.dev)
        return self.buf.data_ptr()


def _scratch(dev, stream):
    """The scratch of the calls on a device's stream (its handle; the current one).  Its lock keeps the kernels of
    two threads' calls on one stream from alternating: one call's would overwrite what the other's still read.  A
    recorded graph gets a buffer of its own, in the graph's memory: it runs at any time, on any stream, and a kept
    buffer may be replaced by a larger one."""
    if _capturing(stream):
        return _Scratch(dev)
    key = (dev.index, stream)
    s = _ws_cache.get(key)
    if s is None:
        with _ws_lock:
            s = _ws_cache.setdefault(key, _Scratch(dev))
    return s


def release_workspace():
    with _ws_lock:
        _ws_cache.clear()


def _capturing(stream) -> bool:
    """Whether the current stream (its handle) records a graph; the null stream cannot."""
    return stream != 0 and torch._C._cuda_isCurrentStreamCapturing()


_marks: dict = {}  # (device, stream) -> event behind the latest table made there


class _Made:
    """Where the kernels that made a table were enqueued, and what other streams need before they read it."""

    __slots__ = ("dev", "stream", "event", "streams")

    def __init__(self, dev, stream):
        self.dev, self.stream = dev, stream
        self.streams = {stream}  # streams that may use the table and its memory in their own order
        # one event per stream, recorded again by each table (waiting for a later table too is no harm), without a
        # system-wide fence: writing the caches back would cost the first call on new weights 30 us
        lib = _lib.load()
        self.event = _marks.get((dev.index, stream))  # None once it is known to have passed
        if self.event is None:
            e = ctypes.c_void_p()
            with torch.cuda.device(dev):
                _lib.check(lib.cvn_event_create(ctypes.byref(e)), "transfer table")
            self.event = _marks.setdefault((dev.index, stream), e)
        _lib.check(lib.cvn_event_record(self.event, stream), "transfer table")

    def join(self, table, stream):
        """Orders the current stream (its handle) after the making of the table, and the release of the table's
        memory after what that stream has enqueued by then.  False while the making stream records a graph."""
        if self.event is not None:
            rc = _lib.load().cvn_event_join(self.event, self.stream, stream)
            if rc == _lib.CVN_ERR_UNSUPPORTED:
                return False
            _lib.check(rc, "transfer table")
        table.record_stream(torch.cuda.current_stream(self.dev))
        self.streams.add(stream)
        return True

    def finish(self):
        """Waits on the host: a stream that records a graph cannot wait for an event from outside it."""
        if self.event is not None:
            _lib.check(_lib.load().cvn_event_wait(self.event, self.stream), "transfer table")
            self.event = None


class _Entry(tuple):
    """(table, memory of psf and bias), with `made` (None without a stream)."""


class TableCache:
    """LRU cache of transfer tables, the counterpart of the reference's OTF cache (converse2d.cpp:52-102).

    Key: the psf and bias tensors (data pointer, strides and version counter), eps, the geometry, the route
    (which fixes the table's layout) and the device.  Entries hold the memory of psf and bias (detached
    views: a parameter itself drops its memory when `.data` is assigned, as Module.to does, and keeps its
    version), so a cached address cannot be reused by another tensor while the entry lives.  An in-place update
    (optimizer step, load_state_dict) bumps the version and misses; the entry of the older version is
    dropped then, so updates leave no dead tables behind.  Writes through `.data` (p.data.copy_(...),
    p.data.mul_(...)) do not bump the version counter: call torch.ops.converse2d.clear_cache() after such
    a write, as with the reference's cache, which keys on the data pointer alone.

    Callers cache only tables that can be hit again (see `cacheable`).  Bounded by the reference's
    64 entries and by bytes.

    Tables are read on any stream: a hit on another stream than the one that made the table waits for it there.
    A table made while its stream records a graph exists once the graph has run, so it is not kept; one from
    before that the graph reads stays until the psf's memory is released (the graph goes on reading it after an
    update of the parameters and clear_cache: record it again then).  At most max_entries tables stay that way;
    past that, a graph makes its own."""

    def __init__(self, max_entries=64, max_bytes=4 << 30):
        from collections import OrderedDict

        self.entries = OrderedDict()
        self._lock = threading.RLock()
        self.latest = {}  # key without version counters -> full key
        self.max_entries = max_entries
        self.max_bytes = max_bytes
        self.bytes = 0
        self.hits = 0
        self.misses = 0
        self.recorded = []  # (psf storage, table) read by recorded graphs

    @staticmethod
    def _stem(key):
        return key[:2] + key[3:4] + key[5:]

    def _keep_recorded(self, e):  # caller holds self._lock
        self.recorded = [r for r in self.recorded if not r[0].expired()]
        if any(t is e[0] for _, t in self.recorded):
            return True
        if len(self.recorded) >= self.max_entries or sum(t.numel() for _, t in self.recorded) > self.max_bytes:
            return False
        self.recorded.append((StorageWeakRef(e[1][0].untyped_storage()), e[0]))
        return True

    def _usable(self, e, stream):  # caller holds self._lock
        if _capturing(stream):
            e.made.finish()
            return self._keep_recorded(e)
        return stream in e.made.streams or e.made.join(e[0], stream)

    def get(self, key, stream=None):
        """The table of `key` or None.  stream: the current stream's handle, where the table is to be read."""
        with self._lock:
            e = self.entries.get(key)
            if e is None or not (e.made is None or stream is None or self._usable(e, stream)):
                self.misses += 1
                return None
            self.entries.move_to_end(key)
            self.hits += 1
            return e[0]

    def _drop(self, key):  # caller holds self._lock
        t, _ = self.entries.pop(key)
        self.bytes -= t.numel()
        stem = self._stem(key)
        if self.latest.get(stem) == key:
            del self.latest[stem]

    def put(self, key, table, refs, stream=None):
        """Keeps `table`.  stream: the current stream's handle, where its kernels have been enqueued."""
        if stream is not None and _capturing(stream):
            return
        e = _Entry((table, tuple(t.detach() for t in refs)))
        e.made = None if stream is None else _Made(table.device, stream)
        with self._lock:
            old = self.latest.get(self._stem(key))
            if old is not None and old in self.entries:
                self._drop(old)  # the same tensors at an older version: never hit again
            prev = self.entries.pop(key, None)
            if prev is not None:  # another thread built the same table meanwhile: keep one copy
                self.bytes -= prev[0].numel()
            self.entries[key] = e
            self.latest[self._stem(key)] = key
            self.bytes += table.numel()
            while self.entries and (len(self.entries) > self.max_entries or self.bytes > self.max_bytes):
                self._drop(next(iter(self.entries)))

    def clear(self):
        with self._lock:
            self.entries.clear()
            self.latest.clear()
            self.bytes = 0


table_cache = TableCache()


def cacheable(weight, bias) -> bool:
    """Whether a table for (weight, bias) can be hit by a later call: not for inference tensors (no
    version counter; in inference mode they are fresh activations), and not while autograd tracks the
    parameters (an optimizer step changes them before the next call; the reference bypasses its cache
    then, converse2d.cpp:60,68,88)."""
    for t in (weight, bias):
        if t.is_inference() or (torch.is_grad_enabled() and t.requires_grad):
            return False
    return True


def _cache_key(kind, weight, bias, eps, geo, route, dev):
    # with the strides of a view: a transposed or expanded one starts at its base's address and shares its version
    return (kind, weight.data_ptr(), weight._version, bias.data_ptr(), bias._version, float(eps), geo, route,
            dev.index, None if weight.is_contiguous() else weight.stride(),
            None if bias.is_contiguous() else bias.stride())


# os.environ's own mapping: a name that is not set costs 0.6 us through os.environ, which raises for it twice
_ENV = os.environ._data
_plan_memo: dict = {}
_supported_memo: dict = {}  # the library's answers by geometry, as in _plan_memo
_plan_lock = threading.Lock()


def _module_plan(lib, B, C, H, W, pb, kh, kw, s, p):
    """(route, table bytes, scratch bytes) of a module-level call: the library's answers depend only on
    the geometry and CVN_DISABLE_FUSED, so they are asked once per geometry (three queries cost about as
    much host time as a small layer's kernels)."""
    key = (B, C, H, W, pb, kh, kw, s, p, _ENV.get(b"CVN_DISABLE_FUSED"))
    plan = _plan_memo.get(key)
    if plan is None:
        route = lib.cvn_converse2d_route(B, C, H, W, pb, kh, kw, s, p)
        if route < 0:
            _lib.check(route, "converse2d_fused")
        plan = (route, lib.cvn_converse2d_table_bytes(B, C, H, W, pb, kh, kw, s, p, route),
                lib.cvn_converse2d_scratch_bytes(B, C, H, W, pb, kh, kw, s, p, route))
        with _plan_lock:
            if len(_plan_memo) >= 1024:
                _plan_memo.clear()
            _plan_memo[key] = plan
    return plan


def module_route(shape, weight, scale, padding):
    """The library's route (_lib.ROUTE_*) for a module-level call on an input of `shape` (B, C, H, W)."""
    B, C, H, W = (int(v) for v in shape)
    return _module_plan(_lib.load(), B, C, H, W, int(weight.shape[0]), int(weight.shape[2]), int(weight.shape[3]),
                        int(scale), int(padding))[0]


def converse2d_fused(x, weight, bias, scale=1, padding=2, padding_mode="circular", eps=1e-5, act=None,
                     cache=True):
    """Converse2D.forward (util_converse.py:142-192) in one library call: pad, solve, crop.

    x (B,C,H,W); weight (1,C,kh,kw) or (B,C,kh,kw) (per-sample psf, as ConvReverseDataNet);
    bias (1,C,1,1) or (C,).  act='gelu' applies exact GELU to the output on store.  cache=True keeps
    the transfer table of a shared psf (psf batch 1) for reuse while weight and bias are unchanged
    (version-checked); per-sample psfs are activations that change every call and are not cached."""
    lib = _lib.load()
    _need_hip(x, weight, bias)
    if x.dim() != 4:
        raise RuntimeError("x must be (B,C,H,W)")
    B, C, H, W = x.shape
    if weight.dim() != 4 or weight.shape[1] != C or weight.shape[0] not in (1, B):
        raise RuntimeError("weight must be (1,C,kh,kw) or (B,C,kh,kw)")
    if bias.numel() != C:
        raise RuntimeError("bias must hold C values")
    if padding_mode not in _lib.PAD_MODES:
        raise ValueError(f"unknown padding_mode {padding_mode!r}")
    s = int(scale)
    if s < 1:
        raise RuntimeError("scale must be >= 1")
    kh, kw = int(weight.shape[2]), int(weight.shape[3])
    pb = int(weight.shape[0])
    x = x.contiguous()
    if x.data_ptr() % 16:
        x = x.clone()
    dev = x.device
    out = torch.empty((B, C, H * s, W * s), dtype=torch.float32, device=dev)
    if B == 0:
        return out
    p = int(padding)
    route, tb, sb = _module_plan(lib, B, C, H, W, pb, kh, kw, s, p)
    st = _stream(dev)
    key = None
    table = None
    if cache and pb == 1 and cacheable(weight, bias):
        key = _cache_key("module", weight, bias, eps, (C, H, W, kh, kw, s, p), route, dev)
        table = table_cache.get(key, st)
    if table is None:
        wc = weight.contiguous()
        bc = bias.contiguous()
        table = torch.empty(tb, dtype=torch.uint8, device=dev)
        _lib.check(lib.cvn_converse2d_table_f32(wc.data_ptr(), pb, kh, kw, bc.data_ptr(), float(eps), B, C, H, W,
                                                s, p, route, table.data_ptr(), tb, st), "converse2d transfer table")
        if key is not None:
            table_cache.put(key, table, (weight, bias), st)
    ws = _scratch(dev, st)
    with ws.lock:
        rc = lib.cvn_converse2d_apply_f32(
            x.data_ptr(), B, C, H, W, pb, kh, kw, s, p, _lib.PAD_MODES[padding_mode],
            _lib.ACT_GELU if act == "gelu" else _lib.ACT_NONE, route, table.data_ptr(), tb, ws.ptr(sb), sb,
            out.data_ptr(), st)
    _lib.check(rc, "converse2d_fused")
    return out


def supported(x, weight, scale, padding, grad_x=False, grad_weight=False, shape=None) -> bool:
    """Whether the library's forward (and the requested backward) serves this geometry
    (cvn_converse2d_supported); shapes it does not serve go to the PyTorch composition.  shape
    (B, C, H, W) stands in for x's shape when given."""
    lib = _lib.load()
    if weight.dim() != 4 or (shape is None and x.dim() != 4):
        return False
    B, C, H, W = shape if shape is not None else x.shape
    pb, _, kh, kw = weight.shape
    key = (B, C, H, W, pb, kh, kw, int(scale), int(padding), bool(grad_x), bool(grad_weight),
           _ENV.get(b"CVN_DISABLE_FUSED"))
    ok = _supported_memo.get(key)
    if ok is None:
        ok = lib.cvn_converse2d_supported(*key[:9], int(key[9]), int(key[10])) == _lib.CVN_OK
        with _plan_lock:
            if len(_supported_memo) >= 1024:
                _supported_memo.clear()
            _supported_memo[key] = ok
    return ok


def op_supported(x, x0, weight, scale) -> bool:
    """Whether the library's operator path serves this call (its table and scratch queries are
    non-zero for the geometry); shapes it does not serve go to the PyTorch composition.  Malformed
    arguments also answer False here and are then rejected by the composition's checks."""
    if x.dim() != 4 or x0.dim() != 4 or weight.dim() != 4:
        return False
    s = int(scale)
    B, C, h, w = (int(v) for v in x.shape)
    if s < 1 or tuple(x0.shape) != (B, C, h * s, w * s) or weight.shape[0] != 1 or weight.shape[1] != C:
        return False
    if B == 0:
        return True  # an empty batch returns its empty output without a launch (converse2d_op)
    if (s == 1 and x0.data_ptr() == x.data_ptr() and x0.stride() == x.stride() and B > 0
            and supported(x, weight, 1, 0)):
        return True  # served by the module route on the padded plane (converse2d_op)
    lib = _lib.load()
    kh, kw = int(weight.shape[2]), int(weight.shape[3])
    return (lib.cvn_converse2d_op_table_bytes(C, h, w, kh, kw, s) > 0
            and lib.cvn_converse2d_op_scratch_bytes(B, C, h, w, s) > 0)


def converse2d_backward(grad_out, x, weight, bias, scale=1, padding=2, padding_mode="circular", eps=1e-5,
                        need_x=True, need_weight=True, need_bias=True):
    """Gradients of Converse2D.forward (util_converse.py:142-192) in one library call: returns
    (grad_x, grad_weight, grad_bias), None where not requested.  grad_out (B,C,H*s,W*s); weight
    (1 or B, C, kh, kw); bias (1,C,1,1) or (C,)."""
    lib = _lib.load()
    _need_hip(grad_out, x, weight, bias)
    B, C, H, W = x.shape
    s, p = int(scale), int(padding)
    if tuple(grad_out.shape) != (B, C, H * s, W * s):
        raise RuntimeError("grad_out must be (B,C,H*scale,W*scale)")
    if weight.dim() != 4 or weight.shape[1] != C or weight.shape[0] not in (1, B):
        raise RuntimeError("weight must be (1,C,kh,kw) or (B,C,kh,kw)")
    if padding_mode not in _lib.PAD_MODES:
        raise ValueError(f"unknown padding_mode {padding_mode!r}")
    kh, kw = int(weight.shape[2]), int(weight.shape[3])
    pb = int(weight.shape[0])
    dev = x.device
    go = grad_out.contiguous()
    xc = x.contiguous()
    wc = weight.contiguous()
    bc = bias.contiguous()
    gx = torch.empty((B, C, H, W), dtype=torch.float32, device=dev) if need_x else None
    gw = torch.empty((pb, C, kh, kw), dtype=torch.float32, device=dev) if need_weight else None
    gb = torch.empty((C,), dtype=torch.float32, device=dev) if need_bias else None
    if B == 0 or not (need_x or need_weight or need_bias):
        for t in (gw, gb):
            if t is not None:
                t.zero_()
        return gx, gw, gb.reshape(bias.shape) if gb is not None else None
    nb = lib.cvn_converse2d_bwd_workspace(B, C, H, W, pb, kh, kw, s, p)
    if nb == 0:
        _lib.check(_lib.CVN_ERR_ARG, "converse2d_backward")
    ptr = lambda t: t.data_ptr() if t is not None else None  # noqa: E731
    st = _stream(dev)
    ws = _scratch(dev, st)
    with ws.lock:
        rc = lib.cvn_converse2d_bwd_f32(go.data_ptr(), xc.data_ptr(), B, C, H, W, wc.data_ptr(), pb, kh, kw,
                                        bc.data_ptr(), float(eps), s, p, _lib.PAD_MODES[padding_mode], ptr(gx),
                                        ptr(gw), ptr(gb), ws.ptr(nb), nb, st)
    _lib.check(rc, "converse2d_backward")
    return gx, gw, gb.reshape(bias.shape) if gb is not None else None


class Converse2DFunction(torch.autograd.Function):
    """Converse2D.forward with the library's forward and backward kernels (the reference gets its
    gradients from autograd through the composite op, converse2d.cpp:223-227)."""

    @staticmethod
    def forward(ctx, x, weight, bias, scale, padding, padding_mode, eps):
        ctx.save_for_backward(x, weight, bias)
        ctx.cfg = (scale, padding, padding_mode, eps)
        # the parameters change between training steps, so their tables are not cached
        return converse2d_fused(x, weight, bias.reshape(-1), scale, padding, padding_mode, eps, cache=False)

    @staticmethod
    def backward(ctx, grad_out):
        x, weight, bias = ctx.saved_tensors
        s, p, mode, eps = ctx.cfg
        nx, nw, nb = ctx.needs_input_grad[:3]
        gx, gw, gb = converse2d_backward(grad_out, x, weight, bias, s, p, mode, eps, nx, nw, nb)
        return gx, gw, gb, None, None, None, None


def converse2d_train(x, weight, bias, scale=1, padding=2, padding_mode="circular", eps=1e-5):
    """Differentiable Converse2D forward on the HIP kernels (forward and backward)."""
    return Converse2DFunction.apply(x, weight, bias, scale, padding, padding_mode, eps)


def converse2d_op(x, x0, weight, bias, scale, eps=1e-5, cache=True):
    """The reference op (converse2d.cpp:165-209): x padded (B,C,h,w), x0 (B,C,h*s,w*s) arbitrary;
    returns the uncropped (B,C,h*s,w*s) solution.  The op table (OTF and alias-class terms) is cached
    per (psf, bias, eps, geometry) like the reference's OTF (p2o_cached, converse2d.cpp:58-102)."""
    lib = _lib.load()
    composite.check_op_args(x, x0, weight, bias, scale)
    s = int(scale)
    _need_hip(x, x0, weight, bias)
    B, C, h, w = x.shape
    if tuple(x0.shape) != (B, C, h * s, w * s) or weight.shape[1] != C or bias.shape[1] != C:
        raise RuntimeError("shape mismatch between x, x0, weight and bias")
    if (s == 1 and x0.data_ptr() == x.data_ptr() and x0.stride() == x.stride() and B > 0
            and supported(x, weight, 1, 0)):
        # x0 is x, as the reference module passes it at scale 1 (util_converse.py:166): then
        # X0 = Y and the solve is the module's X = Y (conj K + lambda) / (|K|^2 + lambda) on the
        # given (already padded) plane, one forward and one inverse transform instead of two and one
        return converse2d_fused(x, weight, bias.reshape(-1), 1, 0, "constant", eps, cache=cache)
    x, x0 = x.contiguous(), x0.contiguous()
    dev = x.device
    out = torch.empty((B, C, h * s, w * s), dtype=torch.float32, device=dev)
    if B == 0:
        return out
    kh, kw = int(weight.shape[2]), int(weight.shape[3])
    tb = lib.cvn_converse2d_op_table_bytes(C, h, w, kh, kw, s)
    sb = lib.cvn_converse2d_op_scratch_bytes(B, C, h, w, s)
    if tb == 0 or sb == 0:
        _lib.check(lib.cvn_converse2d_op_f32(None, None, B, C, h, w, None, kh, kw, None, float(eps), s, None, None,
                                             0, None), "converse2d_op")
    st = _stream(dev)
    key = None
    table = None
    if cache and cacheable(weight, bias):
        key = _cache_key("op", weight, bias, eps, (C, h, w, kh, kw, s), 0, dev)
        table = table_cache.get(key, st)
    if table is None:
        wc, bc = weight.contiguous(), bias.contiguous()
        table = torch.empty(tb, dtype=torch.uint8, device=dev)
        _lib.check(lib.cvn_converse2d_op_table_f32(wc.data_ptr(), kh, kw, bc.data_ptr(), float(eps), C, h, w, s,
                                                   table.data_ptr(), tb, st), "converse2d op table")
        if key is not None:
            table_cache.put(key, table, (weight, bias), st)
    ws = _scratch(dev, st)
    with ws.lock:
        rc = lib.cvn_converse2d_op_apply_f32(x.data_ptr(), x0.data_ptr(), B, C, h, w, s, table.data_ptr(), tb,
                                             ws.ptr(sb), sb, out.data_ptr(), st)
    _lib.check(rc, "converse2d_op")
    return out


def converse2d_fwd_oneshot(x, weight, bias, scale=1, padding=2, padding_mode="circular", eps=1e-5, act=None):
    """cvn_converse2d_fwd_f32: the whole module-level forward (table and apply) in one library call, on
    the route the library picks, with one caller workspace."""
    lib = _lib.load()
    _need_hip(x, weight, bias)
    B, C, H, W = x.shape
    s, p = int(scale), int(padding)
    kh, kw, pb = int(weight.shape[2]), int(weight.shape[3]), int(weight.shape[0])
    x, wc, bc = x.contiguous(), weight.contiguous(), bias.contiguous()
    if x.data_ptr() % 16:  # the fused route reads rows as 16-byte vectors
        x = x.clone()
    out = torch.empty((B, C, H * s, W * s), dtype=torch.float32, device=x.device)
    nb = lib.cvn_converse2d_fwd_workspace(B, C, H, W, pb, kh, kw, s, p)
    st = _stream(x.device)
    ws = _scratch(x.device, st)
    with ws.lock:
        rc = lib.cvn_converse2d_fwd_f32(x.data_ptr(), B, C, H, W, wc.data_ptr(), pb, kh, kw, bc.data_ptr(), float(eps),
                                        s, p, _lib.PAD_MODES[padding_mode],
                                        _lib.ACT_GELU if act == "gelu" else _lib.ACT_NONE, out.data_ptr(),
                                        ws.ptr(max(nb, 1)), nb, st)
    _lib.check(rc, "converse2d_fwd")
    return out


def layernorm_cf(x, weight, bias, eps):
    """LayerNorm(data_format='channels_first') (util_converse.py:63-68)."""
    lib = _lib.load()
    _need_hip(x, weight, bias)
    x, weight, bias = x.contiguous(), weight.contiguous(), bias.contiguous()
    B, C = x.shape[:2]
    HW = x[0, 0].numel() if B > 0 else 0
    y = torch.empty_like(x)
    _lib.check(lib.cvn_layernorm_cf_f32(x.data_ptr(), B, C, HW, weight.data_ptr(), bias.data_ptr(), float(eps),
                                        y.data_ptr(), _stream(x.device)), "layernorm_cf")
    return y


def _ptrs(keep, *ts):
    """Addresses of contiguous tensors (None for None).  Copies of others go to `keep`, which the caller holds until
    the call has enqueued its kernels: a copy that is dropped before then gives its memory to the next copy or
    output."""
    out = []
    for t in ts:
        if t is not None and not t.is_contiguous():
            t = t.contiguous()
            keep.append(t)
        out.append(None if t is None else t.data_ptr())
    return out


def conv1x1(x, weight, bias=None, act=None, residual=None, res_scale=None, ln=None, out=None):
    """act(W x + b) [then res_scale * . + residual]; nn.Conv2d(cin, cout, 1) semantics.
    ln=(ln_weight, ln_bias, eps) applies channels-first LayerNorm to x first (fused prologue)."""
    lib = _lib.load()
    _need_hip(x, weight, bias, residual, res_scale)
    x = x.contiguous()
    B, Cin, H, W = x.shape
    Cout = weight.shape[0]
    if weight.numel() != Cout * Cin:
        raise RuntimeError("weight does not match input channels")
    y = out if out is not None else torch.empty((B, Cout, H, W), dtype=torch.float32, device=x.device)
    keep = []
    wptr, bptr, rptr, sptr = _ptrs(keep, weight, bias, residual, res_scale)
    a = _lib.ACT_GELU if act == "gelu" else _lib.ACT_NONE
    st = _stream(x.device)
    if ln is None:
        rc = lib.cvn_conv1x1_f32(x.data_ptr(), B, Cin, H * W, wptr, bptr, Cout, a, rptr, sptr, y.data_ptr(), st)
    else:
        rc = lib.cvn_ln_conv1x1_f32(x.data_ptr(), B, Cin, H * W, *_ptrs(keep, *ln[:2]), float(ln[2]), wptr, bptr, Cout,
                                    a, rptr, sptr, y.data_ptr(), st)
    _lib.check(rc, "conv1x1")
    return y


def ln_mlp_residual(x, ln_w, ln_b, ln_eps, w1, b1, w2, b2, res_scale=None, out=None):
    """x + res_scale * (W2 GELU(W1 LN(x) + b1) + b2): ConverseBlock.conv2 plus its residual."""
    lib = _lib.load()
    _need_hip(x, w1, b1, w2, b2, res_scale)
    x = x.contiguous()
    B, C, H, W = x.shape
    keep = []
    y = out if out is not None else torch.empty_like(x)
    lw, lb, w1_, b1_, w2_, b2_, sp = _ptrs(keep, ln_w, ln_b, w1, b1, w2, b2, res_scale)
    rc = lib.cvn_ln_mlp_residual_f32(x.data_ptr(), B, C, H * W, lw, lb, float(ln_eps), w1_, b1_, w1.shape[0], w2_, b2_,
                                     sp, y.data_ptr(), _stream(x.device))
    _lib.check(rc, "ln_mlp_residual")
    return y


TAIL_SHAPES = {(128, 64, 128)}  # (Ct, C, Cmid) of cvn_conv_ln_mlp_residual_f32


def conv_ln_mlp_residual(t, x, w0, b0, ln_w, ln_b, ln_eps, w1, b1, w2, b2, res_scale1=None, res_scale2=None,
                         out=None, head=None, t_act=None):
    """ConverseBlock tail: y' = x + res_scale1 (W0 a(t) + b0); y = y' + res_scale2 (W2 GELU(W1 LN(y') + b1) + b2),
    a(t) = GELU(t) for t_act='gelu' (t the Converse2D output before the block's GELU), else t.
    With head = (ln_w, ln_b, ln_eps, w, b) of the next block, also returns its Converse2D input
    GELU(w LN(y) + b): (y, t_next); otherwise y."""
    lib = _lib.load()
    _need_hip(t, x, w0, b0, w1, b1, w2, b2, res_scale1, res_scale2)
    t = t.contiguous()
    x = x.contiguous()
    B, Ct, H, W = t.shape
    C = x.shape[1]
    y = out if out is not None else torch.empty_like(x)
    act = _lib.ACT_GELU if t_act == "gelu" else _lib.ACT_NONE
    keep = []
    w0_, b0_, s1, lw, lb, w1_, b1_, w2_, b2_, s2 = _ptrs(keep, w0, b0, res_scale1, ln_w, ln_b, w1, b1, w2, b2, res_scale2)
    common = (t.data_ptr(), act, B, Ct, H * W, w0_, b0_, s1, x.data_ptr(), C, lw, lb, float(ln_eps), w1_, b1_,
              w1.shape[0], w2_, b2_, s2, y.data_ptr())
    if head is None:
        _lib.check(lib.cvn_conv_ln_mlp_residual_f32(*common, _stream(x.device)), "conv_ln_mlp_residual")
        return y
    hw, hb, heps, wh, bh = head
    _need_hip(wh, bh)
    hw_, hb_, wh_, bh_ = _ptrs(keep, hw, hb, wh, bh)
    tn = torch.empty((B, wh.shape[0], H, W), device=x.device, dtype=x.dtype)
    _lib.check(lib.cvn_conv_ln_mlp_head_f32(*common, hw_, hb_, float(heps), wh_, bh_, tn.data_ptr(), _stream(x.device)),
               "conv_ln_mlp_head")
    return y, tn


def copy_(dst, src):
    """Plain device copy through the library (HBM calibration kernel)."""
    lib = _lib.load()
    _need_hip(dst, src)
    _lib.check(lib.cvn_copy_f32(src.data_ptr(), dst.data_ptr(), src.numel(), _stream(src.device)), "copy")
    return dst
