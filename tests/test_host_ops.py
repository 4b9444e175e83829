"""The ops' native host path (checks and launches in C++) against their Python path.

The native path may only take calls that the Python path would run, and must launch the same thing: on the GPU every
form below runs both ways and gives the same bytes.  Forms that it must leave alone (contract violations, CPU
tensors, subclasses, other streams before their workspace exists, capture, installed profiling providers) raise or
run as before.  The CPU tests need the built extension only.
"""

from __future__ import annotations

import sys
import threading
import time
import warnings
from types import SimpleNamespace

import pytest
import torch

from _helpers import require_gpu
from prism_infer import _native
from prism_infer.ops import kv_cache_store, paged_decode, paged_prefill

FP8 = torch.float8_e4m3fn
MODULES = (kv_cache_store, paged_decode, paged_prefill)


@pytest.fixture
def python_path(monkeypatch):
    """A context that switches the modules to their Python path."""

    def run(fn):
        with monkeypatch.context() as m:
            for module in MODULES:
                m.setattr(module, "_HOST", None)
            return fn()

    return run


class _Recorder:
    """The native ops, keeping whether each call was taken."""

    def __init__(self, host):
        assert host is not None, "the native host path is not built"
        self._host, self.taken = host, []

    def __getattr__(self, name):
        def call(*args):
            out = getattr(self._host, name)(*args)
            self.taken.append(out is not None)
            return out
        return call


@pytest.fixture
def native_calls(monkeypatch):
    """Whether the native path took each call since the list was last cleared."""

    recorder = _Recorder(_native.host_ops())
    for module in MODULES:
        monkeypatch.setattr(module, "_HOST", recorder)
    return recorder.taken


def test_cpu_tensors_and_odd_arguments_are_left_to_python():
    host = _native.host_ops()
    if host is None:
        pytest.skip("the extension is not built")
    t = torch.zeros(2, 1, 8)
    c = torch.zeros(4, 1, 8)
    s = torch.zeros(2, dtype=torch.int32)
    assert host.store(t, t, c, c, s, None, None) is None
    assert host.store(None, t, c, c, s, None, None) is None
    assert host.store(t, t, c, c, s, c, None) is None
    assert host.store(t, t) is None
    assert host.decode(t, c, c, s, s, 1.0, None, None, s, 32, {}) is None
    assert host.prefill(t, c, c, s, s, s, 1, 1, 1.0, None, None, {}) is None


def test_an_extension_that_does_not_load_leaves_the_python_path(monkeypatch, tmp_path):
    if not _native.available():
        pytest.skip("the library is not built")
    broken = tmp_path / "_host_ops.so"
    broken.write_bytes(b"not a shared object")
    monkeypatch.setattr(_native, "HOST_OPS_PATH", broken)
    monkeypatch.setattr(_native, "_HOST_OPS", None)
    monkeypatch.setattr(_native, "_HOST_OPS_TRIED", False)
    with pytest.warns(RuntimeWarning, match="Python path"):
        assert _native.host_ops() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _native.host_ops() is None


def test_prefill_outcome_buffers_are_made_once_per_stream(monkeypatch):
    """Calls that the native path declines each time (int64 metadata, say) make no buffers after the first."""

    stream, made = SimpleNamespace(cuda_stream=7), []
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: stream)
    monkeypatch.setattr(torch, "full", lambda *a, **k: made.append("status") or object())
    monkeypatch.setattr(torch, "empty", lambda *a, **k: made.append("pinned") or object())
    buffers: dict = {}
    for _ in range(3):
        paged_prefill._add_outcome_buffers(buffers, torch.device("cuda", 0))
    assert made == ["status", "pinned"] and list(buffers) == [(0, 7)]
    kept = buffers[(0, 7)]
    for other in range(8, 8 + paged_prefill._MAX_OUTCOME_STREAMS - 1):
        stream.cuda_stream = other
        paged_prefill._add_outcome_buffers(buffers, torch.device("cuda", 0))
    assert buffers[(0, 7)] is kept and len(buffers) == paged_prefill._MAX_OUTCOME_STREAMS
    stream.cuda_stream = 99
    paged_prefill._add_outcome_buffers(buffers, torch.device("cuda", 0))
    assert list(buffers) == [(0, 99)]


def _bytes(x):
    return x.contiguous().view(torch.uint8).cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("cache", ["scaled", "unit", "dense"])
def test_store_both_paths(python_path, native_calls, dtype, cache):
    require_gpu()
    _native.device_lib(torch.device("cuda", 0))  # (the first call of a process loads the kernels from Python)
    g = torch.Generator().manual_seed(5)
    key, value = (torch.randn(33, 6, 128, generator=g).to(dtype).cuda()[:, 1:5].contiguous() for _ in range(2))
    packed = torch.randn(33, 3 * 512, generator=g).to(dtype).cuda()
    slots = torch.randperm(64, generator=g)[:33].to(torch.int32).cuda()
    slots[4] = -1
    for k, v in ((key, value), (packed[:, :512].view(33, 4, 128), packed[:, 512:1024].view(33, 4, 128)),
                 (key[:0], value[:0])):
        out = []
        for native in (True, False):
            for shape in ((4, 16, 4, 128), (64, 4, 128)):
                kc = torch.zeros(shape, device="cuda").to(dtype if cache == "dense" else FP8)
                vc = kc.clone()
                scales = [torch.zeros(shape[:-1], device="cuda") for _ in range(2)] if cache == "scaled" else [None] * 2
                call = lambda: kv_cache_store.store_kvcache(k, v, kc, vc, slots[:k.shape[0]], *scales)  # noqa: E731
                native_calls.clear()
                call() if native else python_path(call)
                assert native_calls == ([k.shape[0] > 0] if native else [])
                out.append([_bytes(x).flatten() for x in (kc, vc, *scales) if x is not None])
        for other in out[1:]:
            assert all(torch.equal(a, b) for a, b in zip(out[0], other))


def _decode_case(dtype, cache, batch=3, hkv=4, groups=2, page=32, width=4):
    g = torch.Generator().manual_seed(9)
    pool = batch * width + 1
    q = torch.randn(batch, hkv * groups, 128, generator=g).to(dtype).cuda()
    k, v = ((torch.randn(pool, page, hkv, 128, generator=g) * 2).to(cache).cuda() for _ in range(2))
    ks, vs = ((torch.rand(pool, page, hkv, generator=g) * 0.2).cuda() for _ in range(2))
    tables = torch.randperm(pool, generator=g)[:batch * width].to(torch.int32).view(batch, width).cuda()
    lens = torch.tensor([page * width, 1, 70], dtype=torch.int32).cuda()
    return q, k, v, tables, lens, ks, vs


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,cache", [(torch.bfloat16, FP8), (torch.float16, FP8), (torch.float32, FP8),
                                         (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)])
def test_decode_both_paths(python_path, native_calls, dtype, cache):
    require_gpu()
    q, k, v, tables, lens, ks, vs = _decode_case(dtype, cache)
    bound = torch.tensor(60, dtype=torch.int32, device="cuda")
    wide = torch.cat([q, q], dim=1)[:, ::2]
    forms = [dict(), dict(max_context_len=bound), dict(max_context_len=bound.view(1, 1)), dict(block_n=64)]
    if cache == FP8:
        forms += [dict(k_scale_cache=ks, v_scale_cache=vs)]
    for qq, tt in ((q, tables), (wide, tables), (q, tables.t().contiguous().t()), (q[:2], tables)):
        for form in forms:
            call = lambda: paged_decode.paged_decode_attention(qq, k, v, tt, lens, 0.1, **form)  # noqa: E731
            first = call()
            native_calls.clear()
            native, python = call(), python_path(call)
            assert native_calls == [True]
            assert native.stride() == python.stride() and native.dtype == python.dtype
            assert torch.equal(_bytes(native), _bytes(python)) and torch.equal(_bytes(first), _bytes(python))
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        twice = [paged_decode.paged_decode_attention(q, k, v, tables, lens, 0.1) for _ in range(2)]
    other.synchronize()
    python = python_path(lambda: paged_decode.paged_decode_attention(q, k, v, tables, lens, 0.1))
    assert all(torch.equal(_bytes(x), _bytes(python)) for x in twice)


@pytest.mark.gpu
def test_bad_calls_raise_as_in_python(python_path):
    require_gpu()
    q, k, v, tables, lens, ks, vs = _decode_case(torch.bfloat16, FP8)
    good = dict(k_scale_cache=ks, v_scale_cache=vs)
    paged_decode.paged_decode_attention(q, k, v, tables, lens, 0.1, **good)
    bad = [lambda: paged_decode.paged_decode_attention(q[:, :3], k, v, tables, lens, 0.1, **good),
           lambda: paged_decode.paged_decode_attention(q, k, v, tables.long(), lens, 0.1, **good),
           lambda: paged_decode.paged_decode_attention(q, k, v, tables[:2], lens, 0.1, **good),
           lambda: paged_decode.paged_decode_attention(q, k, v, tables, lens, 0.1, k_scale_cache=ks),
           lambda: paged_decode.paged_decode_attention(q, k, v, tables, lens, 0.1, block_n=48, **good),
           lambda: paged_decode.paged_decode_attention(q, k, v[..., :64], tables, lens, 0.1, **good),
           lambda: paged_decode.paged_decode_attention(q, k, v, tables, lens.cpu(), 0.1, **good),
           lambda: kv_cache_store.store_kvcache(q, q, k, v, lens, ks, vs),
           lambda: kv_cache_store.store_kvcache(q[:, :4], q[:, :4], k, v, lens.long(), ks, vs),
           lambda: kv_cache_store.store_kvcache(q[:, :4], q[:, :4], k, v, lens, ks, None)]
    for call in bad:
        with pytest.raises((ValueError, RuntimeError)) as native:
            call()
        with pytest.raises(type(native.value)) as python:
            python_path(call)
        assert str(native.value) == str(python.value)


@pytest.mark.gpu
def test_store_keeps_its_profile_region():
    require_gpu()
    from prism_infer import observability

    seen = []

    class Region:
        def __init__(self, name, **kwargs):
            seen.append(name)

        def __enter__(self):
            return self

        def __exit__(self, *exc):
            return False

    q, k, v, _, lens, ks, vs = _decode_case(torch.bfloat16, FP8)
    key = q[:, :4].contiguous()
    kv_cache_store.store_kvcache(key, key, k, v, lens, ks, vs)
    observability.install_performance_provider(profile_region_provider=Region, profile_session_provider=lambda: None)
    try:
        kv_cache_store.store_kvcache(key, key, k, v, lens, ks, vs)
    finally:
        observability._reset_performance_providers()
    assert seen == ["attention.kv_store.hip_scaled_fp8"]


@pytest.mark.gpu
def test_prefill_both_paths_errors_and_threads(python_path, native_calls):
    require_gpu()
    _, k, v, tables, _, ks, vs = _decode_case(torch.bfloat16, FP8)
    q = torch.randn(40, 8, 128, device="cuda").to(torch.bfloat16)
    context = SimpleNamespace(block_tables=tables, context_lens=torch.tensor([128, 5, 70], dtype=torch.int32).cuda(),
                              cu_seqlens_q=torch.tensor([2, 22, 27, 37], dtype=torch.int32).cuda())
    call = lambda c=context: paged_prefill.paged_prefill_attention(  # noqa: E731
        q, k, v, c, num_heads=8, num_kv_heads=4, scale=0.1, k_scale_cache=ks, v_scale_cache=vs)
    first = call()
    native_calls.clear()
    native, python = call(), python_path(call)
    assert native_calls == [True]
    assert native.shape == python.shape == (35, 8, 128)
    assert torch.equal(_bytes(native), _bytes(python)) and torch.equal(_bytes(first), _bytes(python))
    # a bad sequence raises its message, and the next good call is unaffected
    broken = SimpleNamespace(**{**vars(context), "context_lens": torch.tensor([128, 4, 70], dtype=torch.int32).cuda()})
    for _ in range(2):
        with pytest.raises(RuntimeError, match="query=5 context=4"):
            call(broken)
        assert torch.equal(_bytes(call()), _bytes(python))
        assert torch.equal(_bytes(call()), _bytes(python))
    results = []

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            results.extend(_bytes(call()) for _ in range(5))

    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 15 and all(torch.equal(r, _bytes(python)) for r in results)


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["store", "decode", "step"])
def test_other_threads_run_during_launches(native_calls, op):
    """A launch may wait for room in the queue: the native path gives up the GIL over it, as ctypes does.

    The interpreter's own switching is off meanwhile, so another thread advances only where a call lets it.
    """

    require_gpu()
    from prism_infer.engine.decode_attention import PagedKVDecodeAttention, pack_decode_metadata

    q, k, v, tables, lens, ks, vs = _decode_case(torch.bfloat16, FP8)
    key = q[:, :4].contiguous()
    layer = PagedKVDecodeAttention(8, 4, 128, 0.1)
    layer.k_cache, layer.v_cache, layer.k_scale_cache, layer.v_scale_cache = k, v, ks, vs
    meta = pack_decode_metadata([5, 77, 400], [6, 70, 33], tables.cpu(), device="cuda")
    bound = torch.tensor(60, dtype=torch.int32, device="cuda")
    call = {"store": lambda: kv_cache_store.store_kvcache(key, key, k, v, lens, ks, vs),
            "decode": lambda: paged_decode.paged_decode_attention(q, k, v, tables, lens, 0.1, max_context_len=bound),
            "step": lambda: layer(q, key, key, meta)}[op]
    call()
    call()
    torch.cuda.synchronize()
    passes, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            passes[0] += 1
            time.sleep(0)

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    thread.start()
    try:
        sys.setswitchinterval(1000.0)
        before = passes[0]
        for _ in range(20000):
            call()
        ran = passes[0] - before
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        thread.join()
        torch.cuda.synchronize()
    print(f"{op}: {ran} passes of another thread in 20000 calls", flush=True)
    assert ran > 1000  # (with the GIL held the calls let 2 to 19 passes through, without it 285000 to 460000)
