"""GPU prefill over caches whose tokens lie far apart (page-major storage), near the 2 GiB that a page's rows may span.

Pages of 16, 32 and 48 tokens: a 64-key tile covers several of them, so rows counted from the tile's start, not from
their page's, would leave the 32-bit offsets.  The outputs are those of the same pages in a dense cache, byte for byte.
"""

from __future__ import annotations

import pytest
import torch

from _helpers import require_gpu
from test_gpu_prefill import _case, _run

pytestmark = pytest.mark.gpu

STRIDE_LIMIT = 2**31 - 1 - 128


def _spread(t, ids, token_stride):
    """The pages of `t` [pages, page, ...] at the block ids `ids` of a cache with that stride (elements) between tokens."""

    page, rest = t.shape[1], t[0, 0].numel()
    blocks = token_stride // rest
    flat = torch.empty(page * token_stride, dtype=t.dtype, device="cuda")
    inner = (128, 1) if t.dim() == 4 else (1,)
    view = flat.as_strided((blocks, *t.shape[1:]), (rest, token_stride, *inner))
    view.view(torch.uint8)[ids.cuda()] = t.cuda().view(torch.uint8) if t.dim() == 4 else t.cuda().view(torch.uint8)
    return view


@pytest.mark.parametrize("page,groups,kv", [(16, 8, 1), (16, 4, 2), (32, 1, 1), (48, 8, 1)])
@pytest.mark.parametrize("scaled", [True, False])
def test_wide_token_strides(page, groups, kv, scaled):
    require_gpu()
    c = _case(20270500 + page, [(40, 200), (17, 61)], num_heads=groups * kv, num_kv_heads=kv, page=page, scaled=scaled)
    want = _run(c)
    rest = kv * 128
    stride = STRIDE_LIMIT // (page - 1) // rest * rest  # the widest that the op takes
    ids = torch.arange(c["k"].shape[0]) * (stride // rest // c["k"].shape[0])
    far = dict(c)
    far["tables"] = torch.where(c["tables"] >= 0, ids[c["tables"].clamp(min=0).long()].int(), c["tables"])
    far["k"], far["v"] = (_spread(c[n], ids, stride) for n in ("k", "v"))
    if scaled:
        wide = (2**31 // 4 - 1) // (page - 1) // kv * kv
        blocks = far["k"].shape[0]
        far["ks"], far["vs"] = (_spread(c[n], ids, wide)[:blocks] for n in ("ks", "vs"))
        assert far["ks"].shape == far["k"].shape[:-1]
    got = _run(far)
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
