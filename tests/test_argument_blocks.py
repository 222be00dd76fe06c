"""Argument blocks packed as bytes hold what the ctypes structures of the C interface hold, field by field (CPU)."""
import ctypes as C

import pytest

from nha_amd import _lib

BLOCKS = [(_lib.pack_prefill, _lib.NhaPrefillArgs), (_lib.pack_prefill_bwd, _lib.NhaPrefillBwdArgs),
          (_lib.pack_hybrid_prologue, _lib.NhaHybridPrologueArgs), (_lib.pack_ring_fill, _lib.NhaRingFillArgs),
          (_lib.pack_decode, _lib.NhaDecodeArgs)]


@pytest.mark.parametrize("pack,cls", BLOCKS, ids=[c.__name__ for _, c in BLOCKS])
def test_packed_block_is_the_structure(pack, cls):
    values, want = [], cls()
    for name, t in cls._fields_:
        n = getattr(t, "_length_", 1)
        new = [len(values) + 1 + i for i in range(n)]
        setattr(want, name, t(*new) if n > 1 else new[0])
        values += new
    assert pack(*values) == bytes(want)
    assert pack(*[0] * len(values)) == bytes(cls())          # NULL is 0


@pytest.mark.parametrize("x", [0, -1, 2**31 - 1, 2**31, -2**31 - 1, 2**63 - 1, 1 << 70])
def test_whole_numbers_out_of_range_wrap_as_in_a_ctypes_field(x):
    a = _lib.NhaPrefillArgs()
    a.wl = x
    assert _lib.i32(x) == a.wl


@pytest.mark.parametrize("x", [0.125, 0.1, 1e300, -1e300, float("inf")])
def test_floats_out_of_range_are_infinite_as_in_a_ctypes_field(x):
    a = _lib.NhaPrefillArgs()
    a.scale = x
    assert _lib.f32(x) == a.scale
