"""The decode step's one launch (store inside the split-K kernel) against the two ops, byte for byte.

Forms: scaled FP8 and 16-bit caches, bf16 and f16, GQA groups 1 to 16, pages of 32 to 256 tokens, batches up to the
64 slots a wave holds and grids up to a workgroup per CU, and above (two launches); contexts that end on a tile's first and last row, one-token and empty
ones; slots that are skipped (-1, past the cache), that lie in another sequence's pages (which must then see the new
row, as after a store) and in nobody's.  Old bytes under the new rows are NaN codes, so a row taken from memory too
early cannot pass unnoticed.  The split-K family is forced, the native call must take the step, and a captured step
must be the number of launches that is meant, so that no case passes without the kernel that it is for.
"""

from __future__ import annotations

import ctypes
from pathlib import Path

import pytest
import torch

from _helpers import require_gpu

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn


def _launches(fn) -> int:
    """Nodes of the graph that `fn` captures."""

    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        fn()
    count = ctypes.c_size_t()
    hip = ctypes.CDLL(str(Path(torch.__file__).parent / "lib" / "libamdhip64.so"))
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    return count.value


class _MustTake:
    """The native ops, where every call has to be taken."""

    def __init__(self, host):
        self._host = host

    def __getattr__(self, name):
        def call(*args):
            out = getattr(self._host, name)(*args)
            assert out is not None, f"{name} was left to Python"
            return out
        return call


def _check(batch, hkv, groups, page, width, dtype, scaled, lens, odd_slots=False, view=False, launches=1):
    from prism_infer import _native
    from prism_infer.engine import decode_attention
    from prism_infer.engine.decode_attention import PagedKVDecodeAttention, pack_decode_metadata
    from prism_infer.ops import paged_decode
    from prism_infer.ops.kv_cache_store import store_kvcache

    paged_decode.set_decode_overrides(path="split")  # (restored behind every test)
    assert decode_attention._HOST is not None, "the native host path is not built"
    g = torch.Generator().manual_seed(batch * 131 + hkv * 7 + page + groups)
    pool = batch * width + 3
    tables = torch.randperm(pool, generator=g)[:batch * width].view(batch, width)
    slots = [int(tables[b, max(n - 1, 0) // page]) * page + max(n - 1, 0) % page for b, n in enumerate(lens)]
    if odd_slots:
        free = sorted(set(range(pool)) - set(tables.flatten().tolist()))
        slots[0] = -1
        slots[1] = int(tables[2, 0]) * page + 1       # a row that sequence 2 attends
        slots[3] = pool * page + 5                    # past the cache
        slots[4] = free[0] * page                     # a page nobody reads
        if batch > 8:
            slots[batch - 1] = int(tables[2, 0]) * page + 2   # the last sequence's row is sequence 2's to attend,
            slots[5] = int(tables[batch - 2, 0]) * page + 1   # and a row of the one before it is sequence 5's
    cache = FP8 if scaled else dtype
    shape = (pool, page, hkv, 128)
    k, v = ((torch.randn(shape, generator=g) * 2).to(cache) for _ in range(2))
    for c in (k, v):
        for s in slots:
            if 0 <= s < pool * page:
                c.view(-1, hkv, 128)[s] = float("nan")
    ks, vs = ((torch.rand(shape[:-1], generator=g) + 0.1) for _ in range(2))
    q = torch.randn(batch, hkv * groups, 128, generator=g).to(dtype)
    wide = torch.randn(batch, 2 * hkv * 128, generator=g).to(dtype).cuda()
    if view:  # K and V as views of one packed projection
        new_k, new_v = (wide[:, i * hkv * 128:(i + 1) * hkv * 128].view(batch, hkv, 128) for i in range(2))
    else:
        new_k, new_v = (torch.randn(batch, hkv, 128, generator=g).to(dtype).cuda() for _ in range(2))
    meta = pack_decode_metadata(slots, lens, tables, device="cuda")
    q = q.cuda()
    results = []
    family = _native.lib().prism_paged_decode_kernel_family(batch, hkv * groups, hkv, 128, page, width,
                                                            _native.dtype_code(cache))
    assert family == 1
    for fused in (False, True, True):
        caches = [x.cuda() for x in (k, v)] + ([x.cuda() for x in (ks, vs)] if scaled else [None, None])
        if fused:
            layer = PagedKVDecodeAttention(hkv * groups, hkv, 128, 0.09)
            layer.k_cache, layer.v_cache, layer.k_scale_cache, layer.v_scale_cache = caches
            if results[1:]:  # (the stream's workspace exists)
                with pytest.MonkeyPatch.context() as m:
                    m.setattr(decode_attention, "_HOST", _MustTake(decode_attention._HOST))
                    out = layer(q, new_k, new_v, meta)
                assert _launches(lambda: layer(q, new_k, new_v, meta)) == launches
            else:
                out = layer(q, new_k, new_v, meta)
        else:
            store_kvcache(new_k, new_v, caches[0], caches[1], meta.slot_mapping, caches[2], caches[3])
            out = paged_decode.paged_decode_attention(
                q, caches[0], caches[1], meta.block_tables, meta.context_lens, 0.09, k_scale_cache=caches[2],
                v_scale_cache=caches[3], max_context_len=meta.max_context_len)
        results.append([x.contiguous().view(torch.uint8).cpu() for x in (out, *caches) if x is not None])
    assert torch.isfinite(results[0][0].view(dtype).float()).all() or odd_slots
    for other in results[1:]:
        for a, b in zip(results[0], other):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scaled", [True, False])
@pytest.mark.parametrize("hkv,groups,page", [(8, 4, 256), (2, 1, 32), (1, 16, 64), (4, 7, 96)])
def test_fused_step_forms(dtype, scaled, hkv, groups, page):
    require_gpu()
    width = 768 // page
    lens = [1, 32, 33, 64, 257, 700, 768, 0, 31]
    _check(len(lens), hkv, groups, page, width, dtype, scaled, lens)
    _check(len(lens), hkv, groups, page, width, dtype, scaled, lens, odd_slots=True, view=True)


@pytest.mark.parametrize("batch,hkv,width,launches", [
    (1, 8, 5, 1), (2, 8, 5, 1), (63, 2, 5, 1), (64, 2, 5, 1), (65, 2, 5, 2),
    (16, 8, 5, 1), (17, 8, 5, 2),  # chunks of a tile per wave: up to a workgroup per CU (of 256), and above
    (9, 8, 33, 1)])                # more than that, with several tiles per wave
def test_fused_step_batches(batch, hkv, width, launches):
    require_gpu()
    lens = [1 + (37 * b) % 300 + 1700 * (width > 5) for b in range(batch)]
    _check(batch, hkv, 4, 64, width, torch.bfloat16, True, lens, odd_slots=batch > 4, launches=launches)


def test_fused_step_long_contexts_and_replay():
    """Several tiles per wave and many chunks; a captured step follows refilled metadata."""

    require_gpu()
    from prism_infer.engine.decode_attention import PagedKVDecodeAttention, pack_decode_metadata

    _check(2, 8, 4, 256, 80, torch.bfloat16, True, [20000, 9999])
    g = torch.Generator().manual_seed(3)
    tables = torch.randperm(24, generator=g).view(3, 8)
    k, v = ((torch.randn(24, 256, 8, 128, generator=g)).to(FP8).cuda() for _ in range(2))
    ks, vs = ((torch.rand(24, 256, 8, generator=g) + 0.1).cuda() for _ in range(2))
    q, nk, nv = (torch.randn(3, h, 128, generator=g).to(torch.bfloat16).cuda() for h in (32, 8, 8))

    def step(ahead):
        lens = [700 + ahead, 1500 + ahead, 5 + ahead]
        slots = [int(tables[b, (n - 1) // 256]) * 256 + (n - 1) % 256 for b, n in enumerate(lens)]
        return pack_decode_metadata(slots, lens, tables, device="cuda")

    def layer():
        a = PagedKVDecodeAttention(32, 8, 128, 0.09)
        a.k_cache, a.v_cache, a.k_scale_cache, a.v_scale_cache = (x.clone() for x in (k, v, ks, vs))
        return a

    meta, eager, captured = step(0), layer(), layer()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        captured(q, nk, nv, meta)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = captured(q, nk, nv, meta)
    for ahead in range(4):
        meta.copy_(step(ahead))
        graph.replay()
        want = eager(q, nk, nv, step(ahead))
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(captured.k_cache.view(torch.uint8), eager.k_cache.view(torch.uint8))
        assert torch.equal(captured.v_scale_cache, eager.v_scale_cache)
