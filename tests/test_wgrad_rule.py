"""Which weight gradients nha_wgrad takes from the library (host side): the sizes at which it is the faster one; and over how many
ranges of tokens it sums them."""
import ctypes as C

import pytest
import torch

from nha_amd import _lib
from nha_amd.ops import _wgrad_supported


def _call(T, width, outs, dtype=torch.bfloat16):
    row = lambda n: torch.empty(1, n, dtype=dtype).expand(T, n)
    return _wgrad_supported(row(width), [row(o) for o in outs])


@pytest.mark.parametrize("T,width,outs,want", [
    (16384, 1024, [1024], True), (5999, 1024, [1024], False), (6000, 2048, [2048], True), (16384, 2048, [2056], False),
    (16384, 4096, [4096], False), (300, 1024, [1024, 1024, 1024, 256], True), (1, 8, [8, 8], True),
    (1024, 3072, [3072, 768, 768, 512], True), (16384, 4096, [4096, 1024, 1024, 512], False), (300, 4096, [4096] * 3 + [512], False),
    (300, 1024, [1024, 1020], False), (300, 1028, [1024, 1024], False), (300, 1024, [1024] * 5, False)])
def test_sizes(T, width, outs, want):
    assert _call(T, width, outs) == want
    assert not _call(T, width, outs, torch.float32)


@pytest.mark.parametrize("T,width,outs,want", [
    (16384, 1024, [1024], 16), (12000, 1024, [1024], 15), (8192, 1024, [1024], 13), (4096, 1024, [1024, 256, 256, 128], 8),
    (16384, 1024, [1024, 1024, 1024, 256], 4), (16384, 2048, [2048], 4), (16384, 2048, [2048, 512, 512, 256], 2),
    (16384, 3072, [3072, 768, 768, 512], 1), (1000, 1024, [1024, 1024, 1024, 256], 2), (300, 1024, [1024, 1024, 1024, 256], 1), (1, 8, [8], 1)])
def test_token_ranges(T, width, outs, want):
    a = _lib.NhaWgradArgs(n=len(outs), T=T, I=width)
    a.O[:len(outs)] = outs
    assert _lib.load().nha_wgrad_scratch_bytes(C.byref(a)) == want * sum(outs) * width * 4
