"""Register use of compiled kernels, read from the metadata notes of the code objects inside the built libdlt_hip.so (no GPU)."""
import os
import struct

import pytest

from dl_templates_amd import _lib

EM_AMDGPU, SHT_NOTE, NT_AMDGPU_METADATA = 224, 7, 32


@pytest.fixture(scope="module")
def kernels():
    """{mangled name: metadata} of every kernel of the library."""
    msgpack = pytest.importorskip("msgpack")
    if not os.path.exists(_lib.LIB_PATH):
        _lib.build()
    with open(_lib.LIB_PATH, "rb") as f:
        blob = f.read()
    found, pos = {}, blob.find(b"\x7fELF", 4)
    while pos >= 0:
        if struct.unpack_from("<H", blob, pos + 18)[0] == EM_AMDGPU:
            (table,), (size, count) = struct.unpack_from("<Q", blob, pos + 40), struct.unpack_from("<HH", blob, pos + 58)
            for section in range(pos + table, pos + table + size * count, size):
                if struct.unpack_from("<I", blob, section + 4)[0] != SHT_NOTE:
                    continue
                offset, length = struct.unpack_from("<QQ", blob, section + 24)
                note = pos + offset
                while note < pos + offset + length:
                    name, desc, kind = struct.unpack_from("<III", blob, note)
                    at = note + 12 + (name + 3) // 4 * 4
                    if kind == NT_AMDGPU_METADATA:
                        found.update((k[".name"], k) for k in msgpack.unpackb(blob[at:at + desc])["amdhsa.kernels"])
                    note = at + (desc + 3) // 4 * 4
        pos = blob.find(b"\x7fELF", pos + 4)
    return found


def test_tile_window_backward_kernels_spill_nothing(kernels):
    """A spilled register inside their march waits for every staged piece in flight."""
    march = {n: k for n, k in kernels.items() if "swat_bwd_" in n}
    assert len(march) >= 20
    assert {n: k[".vgpr_spill_count"] for n, k in march.items() if k[".private_segment_fixed_size"]} == {}


def test_dq_on_eight_waves_is_built_without_a_mask_only(kernels):
    """flash_backward picks 8 waves of one block for dense calls; under a mask 4 waves run wherever they would."""
    eight = [n for n in kernels if "flashd_bwd_q_kernel" in n and "ELi1ELi64ELi8E" in n]   # <.., NP 1, CK 64, NW 8, MODE, PAD>
    assert eight and not [n for n in eight if "ELi1ELi64ELi8ELi1E" in n]
