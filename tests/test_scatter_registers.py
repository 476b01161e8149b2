"""What the compiler has made of the scattering kernels, as the built library says it: registers that do not fit are spilled to memory, and a load of the
next tile that is spilled is waited for as soon as it is made."""
import re

import pytest

from permutohedral_encoding_amd.build import LIB_PATH


def kernels_of_library():
    """{kernel name: its metadata} from the notes of the device code objects in the library (AMDGPU metadata: msgpack)."""
    msgpack = pytest.importorskip("msgpack")
    blob = open(LIB_PATH, "rb").read()
    found = {}
    for at in (m.start() for m in re.finditer(rb"AMDGPU\x00\x00", blob)):  # the note's name, padded to a multiple of four; size and type stand before it
        size, kind = int.from_bytes(blob[at - 8:at - 4], "little"), int.from_bytes(blob[at - 4:at], "little")
        if kind == 32 and int.from_bytes(blob[at - 12:at - 8], "little") == 7:
            notes = msgpack.unpackb(blob[at + 8:at + 8 + size], strict_map_key=False)
            found.update({k[".name"]: k for k in notes["amdhsa.kernels"]})
    return found


def test_scattering_kernels_keep_a_tile_in_registers():
    scatters = {name: k for name, k in kernels_of_library().items() if re.search(r"backward_table_(both_)?kernel", name)}
    assert len(scatters) >= 7 * 30
    spilled = {name: k[".vgpr_spill_count"] for name, k in scatters.items()}
    # a few addresses, written before the first tile; in workgroups of 1024 threads, seven and eight dimensions, some more of them
    over = {name: n for name, n in spilled.items() if n > (10 if "Li1024E" in name else 4)}
    assert not over
