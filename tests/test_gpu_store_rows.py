"""GPU store into 16- and 32-bit caches (the row path and the scalar path beside it), against torch's casts.

Sizes: one chunk of a row, rows that do not fill a wave, the canonical 8 x 128, rows of several trips; token counts
on both sides of the four-tokens-a-block rule; a view whose rows start off 16 bytes (scalar path).  A cast to the
cache's dtype rounds to nearest even either way, so every finite value is compared bit for bit, and elements of the
cache's own dtype are compared as bits, NaN payloads included.
"""

from __future__ import annotations

import pytest
import torch

from _helpers import require_gpu

pytestmark = pytest.mark.gpu

INTS = {torch.float32: torch.int32, torch.bfloat16: torch.int16, torch.float16: torch.int16}


def _check(in_dtype, cache_dtype, tokens, heads, dim, offset=0):
    from prism_infer.ops.kv_cache_store import store_kvcache

    g = torch.Generator().manual_seed(1000 * heads + dim + tokens)
    rows = []
    for _ in range(2):
        # a packed projection: token rows longer than the K or V part, starting `offset` elements in
        wide = (torch.randn(tokens, heads * dim + 16, generator=g) * 300).to(in_dtype)
        x = wide[:, offset:offset + heads * dim].view(tokens, heads, dim)
        x[0, 0, 0], x[-1, -1, -1] = -0.0, float("inf")
        if in_dtype == cache_dtype:
            x[0, -1, 1] = float("nan")
        rows.append(wide)
    pages, page = -(-tokens // 16) + 2, 16
    slots = torch.randperm(pages * page, generator=g)[:tokens].to(torch.int32)
    if tokens > 4:
        slots[1], slots[3] = -1, pages * page
    caches = [torch.full((pages, page, heads, dim), 7.0, dtype=cache_dtype) for _ in range(2)]
    on_gpu = [c.cuda() for c in caches]
    parts = [w.cuda()[:, offset:offset + heads * dim].view(tokens, heads, dim) for w in rows]
    store_kvcache(parts[0], parts[1], on_gpu[0], on_gpu[1], slots.cuda())
    live = (slots >= 0) & (slots < pages * page)
    for wide, want, got in zip(rows, caches, on_gpu):
        x = wide[:, offset:offset + heads * dim].view(tokens, heads, dim)
        want.view(-1, heads, dim)[slots[live].long()] = x[live].to(cache_dtype)
        assert torch.equal(got.cpu().view(INTS[cache_dtype]), want.view(INTS[cache_dtype]))


@pytest.mark.parametrize("cache_dtype", list(INTS))
@pytest.mark.parametrize("in_dtype", list(INTS))
def test_row_store_dtypes(in_dtype, cache_dtype):
    require_gpu()
    _check(in_dtype, cache_dtype, 37, 8, 128)


@pytest.mark.parametrize("tokens,heads,dim,offset", [(1, 1, 8, 0), (5, 3, 40, 0), (6, 5, 136, 8), (3, 2, 1024, 0),
                                                     (1023, 2, 64, 0), (1027, 4, 128, 8), (9, 3, 5, 0), (9, 8, 128, 1)])
def test_row_store_sizes(tokens, heads, dim, offset):
    require_gpu()
    for in_dtype, cache_dtype in ((torch.bfloat16, torch.bfloat16), (torch.float32, torch.float16)):
        _check(in_dtype, cache_dtype, tokens, heads, dim, offset)
