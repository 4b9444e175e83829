"""Registers of the built kernels: the forms on the main path keep their lanes' values in registers.

Read from the code objects' own notes in the library (the AMDGPU metadata that the compiler writes beside each
kernel).  A spill is a round trip to memory in the inner loop or behind a prologue that every workgroup waits for: the
16-bit decode step with its store cost more than two launches while it spilled 8 registers.
"""

from __future__ import annotations

import re
import struct

import pytest

from prism_infer import _native

msgpack = pytest.importorskip("msgpack")

NOTE_NAME, NT_AMDGPU_METADATA = b"AMDGPU\0\0", 32
# the one-workgroup plan build, and streaming decode of float32 queries over unit-scale caches
MAY_SPILL = ("paged_decode_stream_plan_kernel", "paged_decode_stream_kernelILi0ELb0")


def _kernels() -> dict:
    data = _native.LIB_PATH.read_bytes()
    found, at = {}, data.find(NOTE_NAME)
    while at >= 0:
        name_size, size, kind = struct.unpack_from("<III", data, at - 12)
        if (name_size, kind) == (7, NT_AMDGPU_METADATA):
            note = msgpack.unpackb(data[at + 8:at + 8 + size], raw=False)
            found.update({k[".name"]: k for k in note["amdhsa.kernels"]})
        at = data.find(NOTE_NAME, at + 8)
    return found


def test_main_path_kernels_do_not_spill():
    if not _native.available():
        pytest.skip("the library is not built")
    kernels = _kernels()
    for part in ("paged_decode_split_kernel", "paged_decode_stream_kernel", "paged_prefill_kernel", "kv_store_row_kernel",
                 "compact_held_kernel"):
        assert any(part in name for name in kernels), part
    spilled = {name: k[".vgpr_spill_count"] for name, k in kernels.items()
               if k[".vgpr_spill_count"] and not any(part in name for part in MAY_SPILL)}
    assert not spilled


def test_split_decode_passes_scales_between_lanes_without_lds():
    """Scales that went through LDS in front of the scores cost a decode of one tile per wave 0.4 us of 11."""

    if not _native.available():
        pytest.skip("the library is not built")
    lds = {scaled: {k[".group_segment_fixed_size"] for name, k in _kernels().items()
                    if re.search(rf"paged_decode_split_kernelILi\dELb{scaled}E.*ELb0EEE", name)} for scaled in (0, 1)}
    assert lds[1] and lds[1] <= lds[0], lds
