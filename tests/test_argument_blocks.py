"""Argument blocks packed as bytes hold what the ctypes structures of the C interface hold, field by field (CPU)."""
import ctypes as C

import numpy as np
import pytest
import torch

from nha_amd import _lib, ops

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


@pytest.mark.parametrize("q,k", [((2, 64, 4, 64), (2, 64, 4, 64)), ((128, 4, 64), (2, 64, 4, 64)), ((4, 64), (4, 64))])
@pytest.mark.parametrize("bwd", [False, True])
def test_packed_entries_refuse_tensors_that_are_not_token_major(q, k, bwd):
    """A batch dimension more, and o would have B rows where the kernels write B T (refused before anything is allocated)."""
    q, k, cu = torch.zeros(q), torch.zeros(k), np.array([0, 64, 128], dtype=np.int32)
    with pytest.raises(ValueError, match="token-major"):
        if bwd:
            ops.nha_prefill_bwd(q, k, q, k, k, k, k, q, None, None, q, cu, wl=63, shift=0, scale=0.125)
        else:
            ops.nha_prefill(q, k, q, k, k, k, k, cu, wl=63, shift=0, scale=0.125)
