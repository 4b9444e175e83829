"""When prefill splits keys: scratch is asked for only where parts can pay, which the host weighs as the kernel does.

The shapes and both sides' times, split and not (us): 64 / 8 heads, 400 tokens alone 41.7 and 27.8; 32 / 8 heads, 800
alone 38.2 and 29.7; 267 behind 256 24.7 and 22.7; 33 behind 4096 27.6 and 91.9; 64 / 8 heads, 400 behind 4096 97.8
and 136.4; 8 / 2 heads, 400 behind 512 22.6 and 29.6.
"""

from __future__ import annotations

import pytest

from prism_infer import _native

PAGE = 256


def _scratch(tokens, context, heads, kv):
    if not _native.available():
        pytest.skip("the library is not built")
    return _native.lib().prism_paged_prefill_workspace_bytes(1, tokens, heads, kv, PAGE, -(-context // PAGE))


@pytest.mark.parametrize("tokens,prefix,heads,kv", [(400, 0, 64, 8), (800, 0, 32, 8), (267, 256, 32, 8), (400, 0, 32, 8)])
def test_no_parts_where_their_rows_cost_more_than_the_tiles(tokens, prefix, heads, kv):
    assert _scratch(tokens, tokens + prefix, heads, kv) == 0


@pytest.mark.parametrize("tokens,prefix,heads,kv", [(33, 4096, 32, 8), (400, 4096, 64, 8), (400, 512, 8, 2)])
def test_parts_where_contexts_are_long_and_rows_few(tokens, prefix, heads, kv):
    need = _scratch(tokens, tokens + prefix, heads, kv)
    row = (128 + 2) * 4
    assert need >= 256 + 2 * tokens * heads * row


def test_scratch_is_bounded_by_the_chip():
    """Parts never outnumber the workgroups that fit at once, so neither do their rows, whatever the context."""

    for tokens in (1, 33, 500, 4000):
        for heads, kv in ((8, 8), (32, 8), (64, 8), (4, 1)):
            assert _scratch(tokens, 10**6, heads, kv) <= 256 + 2 * 65536 * (128 + 2) * 4
