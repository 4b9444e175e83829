"""GPU prefill with a block's keys split over workgroups, and the order and query tiles around it.

Short chunks behind long contexts take the split (the workspace query says so); parts may be empty (a one-token
sequence beside a long one) and the scratch may hold anything (NaN here).  Each case runs with the scratch and, by
the entry point that takes none, unsplit, and both are held to the bounds of the other prefill cases against the
fp32-dequantisation oracle.  Merging weighs fp32 partials, so the two agree to the rounding of the bf16 output and
of P (2^-9 each): 2e-2 of the largest output is more than twice that.
"""

from __future__ import annotations

import pytest
import torch

import oracle
from _helpers import require_gpu
from test_gpu_prefill import _case, _want

pytestmark = pytest.mark.gpu


def _run(c, split, parts=None):
    from prism_infer import _native

    lib, dev = _native.device_lib(torch.device("cuda", 0)), torch.device("cuda", 0)
    t = {n: None if c[n] is None else c[n].to(dev) for n in ("q", "k", "v", "ks", "vs", "tables", "lens", "cu")}
    q, batch, width, page = t["q"], t["lens"].numel(), t["tables"].shape[1], t["k"].shape[1]
    out = torch.full_like(q, 77.0)
    status = torch.full((1,), 2**31 - 1, dtype=torch.int32, device=dev)
    need = lib.prism_paged_prefill_workspace_bytes(batch, q.shape[0], c["num_heads"], c["num_kv_heads"], page, width)
    assert need > 0, "the case is meant to be split"
    ws = torch.full((need // 4,), float("nan"), device=dev)
    zero3 = _native.int64s(0, 0, 0)
    scaled = t["ks"] is not None
    args = [q.data_ptr(), _native.dtype_code(q.dtype), _native.strides(q), t["k"].data_ptr(), t["v"].data_ptr(),
            _native.dtype_code(t["k"].dtype), _native.strides(t["k"]), _native.strides(t["v"]),
            t["ks"].data_ptr() if scaled else None, t["vs"].data_ptr() if scaled else None,
            _native.strides(t["ks"]) if scaled else zero3, _native.strides(t["vs"]) if scaled else zero3,
            t["tables"].data_ptr(), _native.strides(t["tables"]), t["lens"].data_ptr(), t["cu"].data_ptr(),
            out.data_ptr(), _native.strides(out), batch, q.shape[0], c["num_heads"], c["num_kv_heads"], 128, page,
            t["k"].shape[0], width, 128 ** -0.5, status.data_ptr()]
    stream = _native.stream_handle(dev)
    if split:
        rc = lib.prism_paged_prefill_ws(*args, ws.data_ptr(), need, None, stream)
    else:
        rc = lib.prism_paged_prefill(*args, stream)
    _native.check(rc, "prefill")
    torch.cuda.synchronize()
    assert status.item() == 2**31 - 1
    if parts is not None:
        parts.append(ws.view(torch.int32)[0].item())  # the parts that the kernel chose
    return out.float().cpu()


def _both(c, label):
    want = _want(c, oracle.prefill_reference_fp32).float()
    mag = max(1.0, want.abs().max().item())
    got = {split: _run(c, split) for split in (True, False)}
    for split, x in got.items():
        err = (x - want).abs()
        assert torch.isfinite(x).all() and err.max().item() < 2e-2 * mag and err.mean().item() < 2e-3 * mag, \
            f"{label} split={split}: max {err.max().item():.3e} mean {err.mean().item():.3e}"
    assert (got[True] - got[False]).abs().max().item() < 2e-2 * mag, label


@pytest.mark.parametrize("heads,kv", [(8, 8), (16, 8), (32, 8), (64, 8), (4, 1), (6, 6)])
def test_split_groups(heads, kv):
    require_gpu()
    _both(_case(20270100 + heads, [(19, 3001), (1, 40), (33, 1300)], num_heads=heads, num_kv_heads=kv),
          f"heads {heads}/{kv}")


@pytest.mark.parametrize("page,qdtype,scaled", [(16, torch.bfloat16, True), (48, torch.float16, True),
                                                (96, torch.bfloat16, False), (192, torch.float16, False),
                                                (64, torch.bfloat16, True)])
def test_split_pages_and_types(page, qdtype, scaled):
    require_gpu()
    _both(_case(20270200 + page, [(1, 1537), (70, 2049), (5, 5)], page=page, qdtype=qdtype, scaled=scaled),
          f"page {page}")


@pytest.mark.parametrize("heads,kv", [(3, 3), (6, 3), (12, 3)])
def test_query_tiles_and_order(heads, kv):
    """Chunks on both sides of the query tiles (128, 64 and 32 tokens), several sequences at one level."""

    require_gpu()
    seqs = [(31, 31), (32, 100), (33, 400), (64, 64), (65, 65), (127, 600), (128, 128), (129, 129), (300, 301)]
    c = _case(20270300 + heads, seqs, num_heads=heads, num_kv_heads=kv, page=64)
    from test_gpu_prefill import _check
    _check(c, f"heads {heads}/{kv}")


def test_parts_follow_the_contexts_and_not_the_tables():
    """One table width (a 4800-token context's) serves all: the kernel weighs the real contexts."""

    require_gpu()
    chosen = {}
    for context in (100, 600, 4700):
        c, parts = _case(20270400, [(70, context), (30, 60)], num_heads=32, num_kv_heads=8, page=64), []
        wide = torch.full((2, 75), -1, dtype=torch.int32)
        wide[:, :c["tables"].shape[1]] = c["tables"]
        c["tables"] = wide
        _run(c, True, parts)
        _both(c, f"context {context}")
        chosen[context] = parts[0]
    assert chosen[100] == 1 and 1 < chosen[600] < chosen[4700], chosen


@pytest.mark.parametrize("qdtype,scaled,page", [(torch.bfloat16, True, 64), (torch.float16, True, 16),
                                                (torch.bfloat16, False, 32), (torch.float16, False, 128)])
@pytest.mark.parametrize("kv", [1, 3, 8])
def test_eight_heads_a_kv_head_by_four_and_by_eight(kv, qdtype, scaled, page):
    """Tables of up to 2048 keys give a workgroup four of the eight heads, wider ones all of them."""

    require_gpu()
    from test_gpu_prefill import _check
    seqs = [(33, 2000), (1, 1), (64, 64), (17, 900)]
    c = _case(20270500 + kv, seqs, num_heads=8 * kv, num_kv_heads=kv, qdtype=qdtype, scaled=scaled, page=page)
    for width in (2048 // page, 2048 // page + 1):
        wide = torch.full((len(seqs), width), -1, dtype=torch.int32)
        n = min(width, c["tables"].shape[1])
        wide[:, :n] = c["tables"][:, :n]
        _check(dict(c, tables=wide), f"{width} pages of {page}")
        _both(dict(c, tables=wide), f"{width} pages of {page}")
