"""GPU prefill: a row's bits do not depend on the query columns of its workgroup that hold no query.

With small scores no tile after the first raises a running max, so a row goes through the same operations whether its
block is full or ends behind it.  Columns without a query that counted as rising would make every tile of their wave
one of maxima, which rounds P differently (and takes longer).
"""

from __future__ import annotations

import pytest
import torch

from _helpers import require_gpu
from test_gpu_prefill import _case
from test_gpu_prefill_split import _run as run_entry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qdtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("groups", [1, 2, 4, 8])
def test_rows_of_a_block_that_ends_early(groups, qdtype):
    require_gpu()
    prefix, full = 1024, 128  # whole blocks for every group size
    c = _case(20270600 + groups, [(full, prefix + full)], num_heads=2 * groups, num_kv_heads=2, qdtype=qdtype)
    c["q"] = c["q"] * 0.05
    want = run_entry(c, False)
    for rows in (1, 8, 31, 33, 40, 65, 100, 127):
        cut = dict(c, q=c["q"][:rows], lens=torch.tensor([prefix + rows], dtype=torch.int32),
                   cu=torch.tensor([0, rows], dtype=torch.int32))
        assert torch.equal(run_entry(cut, False), want[:rows]), rows
