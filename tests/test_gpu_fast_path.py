"""GPU: the native call path (pie_amd/_fast) against the wrappers' general path, over the forms it
takes (ranks, row strides, given outputs, single rows, odd sizes) and forms it hands back (types,
layouts, modes): same bits, same objects for given outputs, same exceptions."""
from __future__ import annotations

import contextlib
import ctypes as C

import pytest
import torch

from pie_amd import _lib, attention, ops
from pie_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _loaded(dev):
    _lib.load()
    assert _lib.fast is not None


def _x(dev, *shape, seed=0):
    return wl.normal(shape, seed + sum(shape)).to(dev)


def _both(monkeypatch, call):
    """call() on the native path (counted) and on the general path."""
    got = call()
    with monkeypatch.context() as m:
        m.setattr(_lib, "fast", None)
        want = call()
    torch.cuda.synchronize()
    got, want = (r if isinstance(r, tuple) else (r,) for r in (got, want))
    for g, w in zip(got, want):
        assert g.shape == w.shape and g.dtype == w.dtype and g.stride() == w.stride()
        assert torch.equal(g.view(torch.int16), w.view(torch.int16))


def _both_refuse(monkeypatch, call):
    """call() raises the same exception with the native path and without it."""
    with pytest.raises(Exception) as got:
        call()
    with monkeypatch.context() as m:
        m.setattr(_lib, "fast", None)
        with pytest.raises(Exception) as want:
            call()
    assert got.type is want.type and str(got.value) == str(want.value)


def _rows(dev, kind, n, cols):
    if kind == "2d":
        return _x(dev, n, cols)
    if kind == "1d":
        return _x(dev, cols)
    if kind == "4d":
        return _x(dev, 2, 1, n, cols)
    if kind == "padded":  # rows of a wider tensor
        return _x(dev, n, cols + 24)[:, 8:8 + cols]
    if kind == "strided":  # inner stride 2: a copy is needed
        return _x(dev, n, 2 * cols)[:, ::2]
    return _x(dev, n, 3, cols).transpose(0, 1)  # rows of no single stride


@pytest.mark.parametrize("kind", ["2d", "1d", "4d", "padded", "strided", "transposed"])
@pytest.mark.parametrize("n,cols", [(1, 64), (3, 2880), (5, 1001)])
def test_row_ops(dev, monkeypatch, kind, n, cols):
    print(f"fast rows {kind} {n} {cols}", flush=True)
    x, r = _rows(dev, kind, n, cols), _rows(dev, kind, n, cols) * 2
    w = _x(dev, cols, seed=3)
    for gemma in (False, True):
        f = ops.gemma_rms_norm if gemma else ops.rmsnorm
        _both(monkeypatch, lambda: f(x, w, 1e-5))
        f2 = ops.gemma_add_rms_norm if gemma else ops.add_rms_norm
        _both(monkeypatch, lambda: f2(x, r, w))
        new = lambda: torch.empty(x.shape, dtype=torch.bfloat16, device=dev)
        _both(monkeypatch, lambda: f2(x, r, w, 1, out=new(), residual_out=new()))
    out = torch.empty(x.shape, dtype=torch.bfloat16, device=dev)
    assert ops.rmsnorm(x, w, 1e-5, out=out) is out
    wide = torch.empty((*x.shape[:-1], cols + 1), dtype=torch.bfloat16, device=dev)
    for f in (lambda: ops.rmsnorm(x, w[1:]), lambda: ops.rmsnorm(x.float(), w), lambda: ops.rmsnorm(x, w.cpu()),
              lambda: ops.rmsnorm(x, w, 1e-5, out=wide), lambda: ops.add_rms_norm(x, wide, w),
              lambda: ops.silu_and_mul(wide if cols % 2 == 0 else x), lambda: ops.silu_and_mul(x.cpu())):
        _both_refuse(monkeypatch, f)
    if cols % 2 == 0:
        _both(monkeypatch, lambda: ops.silu_and_mul(x))
        _both(monkeypatch, lambda: ops.gelu_tanh_and_mul(x))
    table = _x(dev, 50, cols)
    for ids in (torch.tensor([0, 49, -1, 50, 7], device=dev, dtype=torch.int32),
                torch.arange(8, device=dev, dtype=torch.int32)[::2], torch.tensor(3, device=dev, dtype=torch.int32)):
        _both(monkeypatch, lambda: ops.embedding(ids, table))
    _both(monkeypatch, lambda: ops.embedding(ids, table[:, 1:]))


@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("as_pair", [False, True])
def test_prologue_and_attention(dev, monkeypatch, layout, as_pair):
    a = wl.attn_batch([40, 0, 700], [1, 1, 1], Hq=8, Hkv=2, D=128, page_size=16, seed=9, layout=layout)
    pb, cache = a["batch"], a["cache"].to(dev)
    t = {n: getattr(pb, n).to(dev) for n in ("qo_indptr", "kv_indptr", "kv_indices", "kv_last_page_len",
                                             "positions", "batch_indices")}
    kv = (cache[:, 0], cache[:, 1]) if as_pair else cache
    qkv = _x(dev, 3, 12 * 128)
    q, k, v = wl.split_qkv(qkv, 8, 2, 128)
    qw, kw = _x(dev, 128, seed=1), _x(dev, 128, seed=2)

    def prologue(**kw_):
        return ops.qk_rms_norm_rope_append(q, k, v, qw, kw, 1e-6, t["positions"], t["batch_indices"], t["positions"],
                                           kv, t["kv_indices"], t["kv_indptr"], t["kv_last_page_len"], layout, **kw_)

    _both(monkeypatch, prologue)
    qo, ko = torch.empty(3, 8, 128, dtype=torch.bfloat16, device=dev), torch.empty(3, 2, 128, dtype=torch.bfloat16,
                                                                                 device=dev)
    r = prologue(q_out=qo, k_out=ko)
    assert r[0] is qo and r[1] is ko
    ws = torch.zeros(32 << 20, dtype=torch.uint8, device=dev)
    d = attention.BatchDecodeWithPagedKVCacheWrapper(ws, layout)
    d.plan(t["kv_indptr"], t["kv_indices"], t["kv_last_page_len"], 8, 2, 128, 16)
    p = attention.BatchPrefillWithPagedKVCacheWrapper(torch.zeros_like(ws), layout)
    p.plan(t["qo_indptr"], t["kv_indptr"], t["kv_indices"], t["kv_last_page_len"], 8, 2, 128, 16, causal=True)
    qs = q.contiguous()
    for w in (d, p):
        for x in (qs, q):
            _both(monkeypatch, lambda: w.run(x, kv))
        out = torch.empty_like(qs)
        assert w.run(qs, kv, out=out) is out
        for bad in (qs[:2], qs.float(), qs.cpu(), qs[:, :, ::2]):
            _both_refuse(monkeypatch, lambda: w.run(bad, kv))


def test_modes_and_subclasses_take_the_general_path(dev):
    """Under a dispatch mode, and for tensor subclasses, the native path declines."""
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    x, w = _x(dev, 4, 64), _x(dev, 64)
    assert _lib.fast.rmsnorm(x, w, 1e-5, None, False) is not None
    with Mode():
        assert _lib.fast.rmsnorm(x, w, 1e-5, None, False) is None
    assert _lib.fast.rmsnorm(x.as_subclass(Sub), w, 1e-5, None, False) is None
    assert _lib.fast.rmsnorm(x, w, "1e-5", None, False) is None
    assert _lib.fast.rmsnorm(x) is None


_ENTRY_POINTS = ("pie_hip_rmsnorm", "pie_hip_gemma_rmsnorm", "pie_hip_fused_add_rmsnorm",
                 "pie_hip_gemma_fused_add_rmsnorm", "pie_hip_silu_and_mul", "pie_hip_gelu_tanh_and_mul",
                 "pie_hip_embedding", "pie_hip_qk_rmsnorm_rope_append", "pie_hip_attention_decode",
                 "pie_hip_attention_prefill_split")


@contextlib.contextmanager
def _native_entry_points_return(rc, calls):
    """The native path's entry points replaced by stubs that record their name and return rc."""
    addr = _lib._addresses(_lib.load())
    stubs = {}
    for n in _ENTRY_POINTS:
        def stub(*args, n=n):
            calls.append(n)
            return rc
        stubs[n] = C.CFUNCTYPE(C.c_int, *_lib.SIGNATURES[n])(stub)
    try:
        _lib.fast.bind({**addr, **{n: C.cast(f, C.c_void_p).value for n, f in stubs.items()}}, _lib._check_rc)
        yield
    finally:
        _lib.fast.bind(addr, _lib._check_rc)


def _one_call_each(dev):
    """(entry point, call) of every op the native path serves; the in-place ones among them."""
    x, r, w = _x(dev, 4, 256), _x(dev, 4, 256, seed=1), _x(dev, 256, seed=2)
    a = wl.attn_batch([40, 0, 700], [1, 1, 1], Hq=8, Hkv=2, D=128, page_size=16, seed=9)
    pb, cache = a["batch"], a["cache"].to(dev)
    t = {n: getattr(pb, n).to(dev) for n in ("qo_indptr", "kv_indptr", "kv_indices", "kv_last_page_len",
                                             "positions", "batch_indices")}
    q, k, v = wl.split_qkv(_x(dev, 3, 12 * 128), 8, 2, 128)
    qw, kw = _x(dev, 128, seed=1), _x(dev, 128, seed=2)
    ws = lambda: torch.zeros(32 << 20, dtype=torch.uint8, device=dev)
    d = attention.BatchDecodeWithPagedKVCacheWrapper(ws(), "NHD")
    d.plan(t["kv_indptr"], t["kv_indices"], t["kv_last_page_len"], 8, 2, 128, 16)
    p = attention.BatchPrefillWithPagedKVCacheWrapper(ws(), "NHD")
    p.plan(t["qo_indptr"], t["kv_indptr"], t["kv_indices"], t["kv_last_page_len"], 8, 2, 128, 16, causal=True)
    qc = q.contiguous()
    return [
        ("pie_hip_rmsnorm", lambda: ops.rmsnorm(x, w)),
        ("pie_hip_gemma_rmsnorm", lambda: ops.gemma_rms_norm(x, w)),
        ("pie_hip_fused_add_rmsnorm", lambda: ops.fused_add_rmsnorm(x, r, w)),
        ("pie_hip_gemma_fused_add_rmsnorm", lambda: ops.gemma_add_rms_norm(x, r, w, residual_out=r)),
        ("pie_hip_silu_and_mul", lambda: ops.silu_and_mul(x)),
        ("pie_hip_gelu_tanh_and_mul", lambda: ops.gelu_tanh_and_mul(x)),
        ("pie_hip_embedding", lambda: ops.embedding(t["positions"], x)),
        ("pie_hip_qk_rmsnorm_rope_append", lambda: ops.qk_rms_norm_rope_append(
            q, k, v, qw, kw, 1e-6, t["positions"], t["batch_indices"], t["positions"], cache, t["kv_indices"],
            t["kv_indptr"], t["kv_last_page_len"], q_out=q, k_out=k)),
        ("pie_hip_attention_decode", lambda: d.run(qc, cache)),
        ("pie_hip_attention_prefill_split", lambda: p.run(qc, cache)),
    ]


def test_a_rejected_launch_raises_and_is_not_repeated(dev):
    """PIE_HIP_ELAUNCH comes after the kernel was handed to the runtime (the error may be an older
    one of the thread): the native path raises it, as the general path does, and runs the op once."""
    for name, call in _one_call_each(dev):
        calls = []
        with _native_entry_points_return(2, calls):
            with pytest.raises(_lib.PieHipError, match=f"{name} failed"):
                call()
        assert calls == [name]


@pytest.mark.parametrize("rc", [1, 3])
def test_a_refusal_before_any_launch_takes_the_general_path(dev, rc):
    """Invalid arguments and busy state are returned before any launch: the general path then runs,
    or refuses, the call."""
    for name, call in _one_call_each(dev):
        calls = []
        with _native_entry_points_return(rc, calls):
            call()
        assert calls == [name]
    torch.cuda.synchronize()
