"""The packed bytes of an expression's C structs against ctypes' own layout of them (CPU)."""
import ctypes as C

import pytest

from packed_amd import _lib
from packed_amd import vexpr as V


@pytest.mark.parametrize("s", [0.5, -0.0, float("inf"), 1e-42, 1e39, -1e300])
def test_struct_bytes(s):
    row = (3, 1, 2, 3, s, -s)
    for cls, pack in ((_lib.VInstr, V._PACK_F32), (_lib.VInstr64, V._PACK_F64)):
        assert pack(*row) == bytes(cls(*row))
    assert V._PACK_SRC(0x123456789A0, 64) == bytes(_lib.VSource(0x123456789A0, 64)) == bytes(_lib.VSource64(0x123456789A0, 64))
    assert C.sizeof(_lib.VInstr) == 24 and C.sizeof(_lib.VInstr64) == 32
