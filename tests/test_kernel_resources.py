"""What the compiler gave the kernels of the built library, from the metadata of its code object (written by this
build's own compiler run): a register that does not fit is kept in scratch memory, which costs the row movers what
they save elsewhere, and static LDS decides how many workgroups a compute unit holds.
"""

from __future__ import annotations

import re

import pytest

from pcie_ep import _native


def unsigned(blob: bytes, at: int) -> int:
    """The MessagePack unsigned integer at `at`."""
    width = {0xCC: 1, 0xCD: 2, 0xCE: 4, 0xCF: 8}.get(blob[at], 0)
    return int.from_bytes(blob[at + 1:at + 1 + width], "big") if width else blob[at]


@pytest.fixture(scope="module")
def kernels():
    """Kernel symbol -> its metadata fields.  A kernel's map is written with its keys in alphabetical order: the
    `.symbol` in front of a `.vgpr_spill_count` and the segment sizes in front of that belong to it."""
    blob = _native.LIBRARY_PATH.read_bytes()
    keys = [".group_segment_fixed_size", ".private_segment_fixed_size", ".symbol", ".vgpr_count", ".vgpr_spill_count"]
    found, fields = {}, {}
    for match in re.finditer(b"|".join(re.escape(bytes([0xD9, len(key)]) + key.encode() if len(key) > 31 else bytes([0xA0 | len(key)]) + key.encode())
                                       for key in keys), blob):
        key = match.group()[match.group().index(b"."):].decode()
        if key == ".symbol":
            size, start = (blob[match.end() + 1], match.end() + 2) if blob[match.end()] == 0xD9 else (blob[match.end()] & 0x1F, match.end() + 1)
            fields["symbol"] = blob[start:start + size].decode()
        else:
            fields[key] = unsigned(blob, match.end())
        if key == keys[-1]:
            found[fields.pop("symbol")] = fields
            fields = {}
    return found


def test_no_kernel_keeps_registers_in_scratch_memory(kernels):
    transport = [symbol for symbol in kernels if "transport_kernel" in symbol]
    assert len(transport) == 8, sorted(kernels)  # wire x whole vectors or ragged x one row or two at a time
    for symbol in transport:
        assert kernels[symbol][".vgpr_count"] > 64 and kernels[symbol][".group_segment_fixed_size"] > 0  # the right fields were read
    spilled = {symbol: fields for symbol, fields in kernels.items() if fields[".vgpr_spill_count"] or fields[".private_segment_fixed_size"]}
    assert not spilled


def test_the_transport_kernels_declare_next_to_no_lds(kernels):
    """A workgroup's scratch and the prologue's tables share the LDS that a launch asks for: four workgroups of the
    largest prologue that then fits (40 960 bytes each of a compute unit's 160 KB) must not be pushed out by what is declared."""
    for symbol, fields in kernels.items():
        if "transport_kernel" in symbol:
            assert fields[".group_segment_fixed_size"] <= 512, symbol
