"""GPU prefill with NaN and infinite inputs: a row that attends to one is NaN, every other row is as without it.

A NaN query element, K byte, key scale or value scale may lie in the first tile, in a settled one (neither first nor
masked), in the tile on the diagonal, or in a prompt that is one tile; the context may be one workgroup's or split over
several.  The oracle in float64 says which outputs are NaN: a masked key has weight 0 there too, except that it
multiplies masked values, so value cases are told from the positions.  Keys whose score is -inf weigh 0, also where
the first tiles hold nothing else.  Finite rows keep the bounds of the other prefill cases.
"""

from __future__ import annotations

import pytest
import torch

import oracle
from _helpers import require_gpu
from test_gpu_prefill import _case, _want
from test_gpu_prefill import _run as run_op
from test_gpu_prefill_split import _run as run_entry

pytestmark = pytest.mark.gpu

PREFIX, CHUNK = 2060, 40
# key positions of sequence 0: first tile, settled tile, the diagonal's tile (rows from 10 on see it)
PLACES = {"first": 3, "settled": 700, "diagonal": PREFIX + 10}


def _make(groups, qdtype, page=256):
    return _case(20270400 + groups, [(CHUNK, PREFIX + CHUNK), (20, 20)], num_heads=2 * groups, num_kv_heads=2, page=page,
                 qdtype=qdtype)


def _slot(c, seq, pos):
    page = c["k"].shape[1]
    return int(c["tables"][seq, pos // page]), pos % page


def _outputs(c):
    return {"op": run_op(c).float(), "split": run_entry(c, True), "one part": run_entry(c, False)}


def _check(c, nan, label):
    """`nan`: which outputs are NaN.  The rest against the oracle."""

    want = _want(c, oracle.prefill_reference_fp32).float()
    ok = ~nan
    mag = max(1.0, want[ok].nan_to_num().abs().max().item())
    for name, got in _outputs(c).items():
        assert torch.equal(torch.isnan(got), nan), f"{label}, {name}: {int((torch.isnan(got) ^ nan).sum())} differ"
        seen = ok & ~torch.isnan(want)
        assert (got - want)[seen].abs().max().item() < 2e-2 * mag, f"{label}, {name}"


@pytest.mark.parametrize("qdtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("groups", [1, 2, 4, 8])
def test_nan_queries(groups, qdtype):
    require_gpu()
    c = _make(groups, qdtype)
    c["q"][5, groups, 77] = float("nan")          # behind the prefix
    c["q"][CHUNK + 7, 0, 0] = float("nan")        # in the one-tile prompt
    if qdtype == torch.float16:
        c["q"][CHUNK + 18, 1, 9] = float("inf")   # infinite scores of both signs
    nan = torch.isnan(_want(c, oracle.prefill_reference_fp32))
    assert nan.any(-1).sum() == 2 + (qdtype == torch.float16)
    _check(c, nan, f"q, groups {groups}")


@pytest.mark.parametrize("page", [256, 16])
@pytest.mark.parametrize("groups,qdtype", [(1, torch.bfloat16), (4, torch.bfloat16), (4, torch.float16)])
@pytest.mark.parametrize("place", list(PLACES))
@pytest.mark.parametrize("what", ["k", "ks"])
def test_nan_keys(what, place, groups, qdtype, page):
    require_gpu()
    c = _make(groups, qdtype, page)
    for seq, pos in ((0, PLACES[place]), (1, 12)):
        blk, off = _slot(c, seq, pos)
        if what == "k":
            c["k"].view(torch.uint8)[blk, off, 1, 33] = 0x7F
        else:
            c["ks"][blk, off, 1] = float("nan")
    nan = torch.isnan(_want(c, oracle.prefill_reference_fp32))
    assert nan.any() and not nan.all()
    _check(c, nan, f"{what} {place}")


@pytest.mark.parametrize("place", list(PLACES))
@pytest.mark.parametrize("groups,qdtype", [(1, torch.bfloat16), (4, torch.float16)])
def test_nan_value_scales(groups, qdtype, place):
    require_gpu()
    c = _make(groups, qdtype)
    pos = PLACES[place]
    c["vs"][(*_slot(c, 0, pos), 1)] = float("nan")
    nan = torch.zeros(CHUNK + 20, 2 * groups, 128, dtype=torch.bool)
    nan[max(pos - PREFIX, 0):CHUNK, groups:] = True
    _check(c, nan, f"vs {place}")


@pytest.mark.parametrize("groups,qdtype", [(1, torch.bfloat16), (4, torch.bfloat16), (4, torch.float16)])
def test_scores_of_minus_infinity_weigh_nothing(groups, qdtype):
    """Negative keys with an infinite scale against positive queries: the first three tiles, and one key further on."""

    require_gpu()
    c = _make(groups, qdtype)
    c["q"] = c["q"].abs() + 0.01
    for pos in (*range(192), 900, PREFIX + 3):
        blk, off = _slot(c, 0, pos)
        c["k"][blk, off] = (-c["k"][blk, off].float().abs() - 0.5).to(c["k"].dtype)
        c["ks"][blk, off] = float("inf")
    nan = torch.isnan(_want(c, oracle.prefill_reference_fp32))
    assert not nan.any()
    _check(c, nan, "-inf")
