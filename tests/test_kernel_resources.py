"""Registers of the compiled kernels, from the metadata that the compiler leaves in the library."""

from __future__ import annotations

import struct

import msgpack
import pytest

from sva_amd import _lib

AMDGPU = 224  # e_machine
NT_AMDGPU_METADATA = 32
SHT_NOTE = 7


def kernels(path) -> dict:
    """{kernel name: its metadata} of every gfx950 code object in the library."""
    data = open(path, "rb").read()
    found, at = {}, data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == AMDGPU:
            shoff = struct.unpack_from("<Q", data, at + 40)[0]
            size, count = struct.unpack_from("<HH", data, at + 58)
            for i in range(count):
                _, kind, _, _, off, length = struct.unpack_from("<IIQQQQ", data, at + shoff + i * size)
                if kind == SHT_NOTE:
                    names, n_desc, note = struct.unpack_from("<III", data, at + off)
                    if note == NT_AMDGPU_METADATA:
                        desc = at + off + 12 + (names + 3) // 4 * 4
                        meta = msgpack.unpackb(data[desc:desc + n_desc])
                        found.update({k[".name"]: k for k in meta["amdhsa.kernels"]})
        at = data.find(b"\x7fELF", at + 4)
    return found


def test_finish_kernels_keep_their_registers():
    """A register too many sends the finish's pointers to memory and back in every phase (fp32 K and V, 1M keys:
    44.0 us a lookup against 37.2)."""
    if not _lib.LIB_PATH.exists():
        pytest.skip("the library is not built")
    finish = {k: v for k, v in kernels(_lib.LIB_PATH).items() if "wide_finish_kernel" in k}
    assert len(finish) == 8  # no verifier (one token, several), six of head_dim and K / V type
    for name, k in finish.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name
