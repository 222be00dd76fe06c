"""Which calls combine their segments in one launch (host side): sequences of up to 16 segments on average, while a launch holds the
workgroups (256 threads each, fewer than 2^32 in all)."""
import ctypes as C

import pytest

from nha_amd import _lib


def _grid(NT, N, H, D, seg_sh):
    rule = _lib.load()["_ZN3nha15state_link_gridEiiiii"]   # nha::state_link_grid
    rule.restype, rule.argtypes = C.c_int64, [C.c_int] * 5
    return rule(NT, N, H, D, seg_sh)


@pytest.mark.parametrize("NT,N,H,D,seg_sh,want", [
    (256, 2, 8, 128, 3, 34 * 8 * 16), (257, 2, 8, 128, 3, 0), (16, 1, 4, 64, 0, 17 * 4 * 8), (17, 1, 4, 64, 0, 0), (6, 1, 4, 256, 0, 7 * 4 * 32),
    (65535, 65535, 16, 128, 3, 0), (65528, 57345, 16, 128, 3, 0), (65528, 57344, 16, 128, 3, (8191 + 57344) * 256), (65520, 57345, 16, 128, 3, (8190 + 57345) * 256),
    (65535, 65535, 56, 64, 3, 0), (65535, 65535, 28, 64, 3, (8191 + 65535) * 28 * 8), (65535, 65535, 6, 256, 3, (8191 + 65535) * 192)])
def test_grid(NT, N, H, D, seg_sh, want):
    assert want < 1 << 24
    assert _grid(NT, N, H, D, seg_sh) == want
