"""CPU check of the built library's own kernels: the permuted stores of 2^13 keep everything in
registers (spilled ones cost the forward transforms of the permuted orders 2 - 8 %)."""
import os
import re
import struct

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def kernels():
    """(name, metadata) of every kernel in the library: the notes of its gfx950 code objects."""
    msgpack = pytest.importorskip("msgpack")
    data = open(os.path.join(ROOT, "packed_amd", "libpcx_gpu.so"), "rb").read()
    for m in re.finditer(b"\x7fELF\x02\x01\x01\x40", data):  # ELF64, little endian, AMDGPU HSA
        elf = memoryview(data)[m.start():]
        phoff, = struct.unpack_from("<Q", elf, 32)
        phsize, phnum = struct.unpack_from("<HH", elf, 54)
        for k in range(phnum):
            kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + k * phsize)
            if kind != 4:  # PT_NOTE
                continue
            namesz, descsz, ntype = struct.unpack_from("<III", elf, off)
            if ntype == 32:  # NT_AMDGPU_METADATA
                at = off + 12 + (namesz + 3) // 4 * 4
                for kernel in msgpack.unpackb(bytes(elf[at:at + descsz]))["amdhsa.kernels"]:
                    yield kernel[".name"], kernel


def test_permuted_stores_of_2_13_stay_in_registers():
    found = {name: k for name, k in kernels() if re.search(r"5k_rowILi13ELi1ELi0ELi1ELi0ELb1ELi[12]ELi0EfLi\d+E", name)}
    assert len(found) == 4  # bit_reversed and unordered, pack 1 and any pack
    for name, k in found.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name
