"""GPU compaction of plans that fit a workgroup's registers, and of the smallest that do not, against the oracle.

Every plan overlaps itself (destinations that are other entries' sources), repeats a source, holds a no-op entry and
entries out of range on either side (skipped).  Sizes: both sides of the 16384-chunk limit and of its half (entries
x chunks of a 128-byte strip), vectors that are no power of two, shorter than a strip, of 4- and 1-byte chunks, long
vectors with few entries (strips that widen) and few rows (fewer workgroups than CUs).
"""

from __future__ import annotations

import pytest
import torch

import oracle
from _helpers import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,slots,vec,retained", [
    (6, 2600, 1024, 2048), (6, 2600, 1024, 2049), (6, 2600, 1024, 1024), (40, 1500, 1024, 1025),
    (2, 9000, 32, 8192), (2, 9000, 32, 8193), (2, 9000, 16, 8192), (150, 300, 48, 200), (150, 300, 1040, 200),
    (4, 5000, 4, 4500), (4, 700, 20, 512), (4, 700, 20, 513), (4, 300, 7, 256), (4, 300, 131, 128), (4, 300, 131, 129),
    (3, 40, 65536, 3), (70, 9, 65552, 1), (1, 5, 16, 2),
])
def test_held_plans(rows, slots, vec, retained):
    require_gpu()
    from prism_infer import _native

    g = torch.Generator().manual_seed(rows + slots + vec + retained)
    cache = torch.randint(0, 256, (1, rows, slots, vec), generator=g, dtype=torch.uint8)
    src = torch.randperm(slots, generator=g)[:retained]
    dst = torch.randperm(slots, generator=g)[:retained]
    if retained >= 128:
        src[3] = src[4]
        dst[5] = src[5]
    want = cache.clone()
    oracle.compact_slots(want, src, dst)
    if retained >= 128:  # entries the oracle refuses and the kernels skip
        extra = torch.tensor([-1, slots, 7, 8])
        src, dst = torch.cat([src, extra]), torch.cat([dst, torch.tensor([1, 2, -5, slots + 9])])
        if retained in (2048, 1024, 8192, 512, 256, 128):
            src, dst = src[4:], dst[4:]  # the plan stays at its limit, without its first entries
            want = cache.clone()
            oracle.compact_slots(want, src[:-4], dst[:-4])
    lib = _native.lib()
    gpu = cache.cuda()
    need = lib.prism_compact_slots_workspace_bytes(rows, slots, vec, src.numel())
    ws = torch.randint(0, 256, (need,), generator=g, dtype=torch.uint8).cuda()
    s, d = src.cuda(), dst.cuda()
    _native.check(lib.prism_compact_slots(gpu.data_ptr(), rows, slots, vec, s.data_ptr(), d.data_ptr(), src.numel(),
                                          ws.data_ptr(), need, _native.stream_handle(gpu.device)), "compact")
    assert torch.equal(gpu.cpu(), want)
