"""Which decode steps use scratch (host side of the C ABI): the ones that spread a (sequence, kv-head) pair over several
workgroups, and the argument block packed in one call."""
import ctypes as C
import os

import pytest

from nha_amd import _lib


def _args(B=2, HQ=8, H=2, D=128, W=200, dtype=_lib.NHA_DTYPE_BF16, mode=_lib.NHA_DECODE_RING, M=64, V=None, q=4096):
    a = _lib.NhaDecodeArgs(mode=mode, dtype=dtype, B=B, HQ=HQ, H=H, K=D, V=V or D, M=M, W=W, scale=1.0, q=q, sq=4096, o=4096)
    return _lib.load().nha_decode_uses_scratch(C.byref(a))


@pytest.mark.parametrize("kw,want", [
    ({}, 1), (dict(B=1, H=1, HQ=8), 1), (dict(W=33), 1), (dict(B=32, H=4, HQ=4), 1), (dict(B=128, H=1, HQ=1), 1),
    (dict(B=128, H=1, HQ=1, W=64), 0), (dict(B=129, H=1, HQ=4), 0), (dict(B=128, H=8, HQ=32, W=1024), 0),
    (dict(B=40, H=3, HQ=3, D=256, W=32), 0), (dict(dtype=_lib.NHA_DTYPE_F32), 0), (dict(q=4098), 0), (dict(D=96), 0),
    (dict(M=32), 0), (dict(V=64), 0), (dict(mode=_lib.NHA_DECODE_LOGITS), 0), (dict(HQ=20), 0), (dict(B=0), 0), (dict(HQ=7), 0)])
def test_sizes(kw, want):
    assert _args(**kw) == want


def test_null():
    assert _lib.load().nha_decode_uses_scratch(None) == 0


def test_packed_block_and_its_scratch():
    fields = _lib.NhaDecodeArgs._fields_
    values = [0.5 if t is C.c_float else i + 1 for i, (_, t) in enumerate(fields)]
    block = _lib.pack_decode(*values)
    assert len(block) == C.sizeof(_lib.NhaDecodeArgs)
    a = _lib.NhaDecodeArgs.from_buffer_copy(_lib.with_scratch(block, 1 << 40, 1 << 33))
    assert [getattr(a, n) for n, _ in fields] == [*values[:-2], 1 << 40, 1 << 33]


def test_struct_layouts_match_the_header(tmp_path):
    """sizeof and offsets of the mirrors that the other layout test does not look at, as the C compiler sees the header."""
    import subprocess
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    probes = [(cls, f) for cls in ("NhaDecodeArgs", "NhaWgradArgs", "NhaRingFillArgs") for f, _ in getattr(_lib, cls)._fields_]
    src = tmp_path / "probe.c"
    src.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "nha_hip.h"\nint main(void) {\n' +
                   "".join(f'printf("%zu %zu\\n", sizeof({c}), offsetof({c}, {f}));\n' for c, f in probes) + "return 0; }\n")
    subprocess.run(["gcc", "-I", os.path.join(root, "include"), str(src), "-o", str(tmp_path / "probe")], check=True)
    lines = subprocess.run([str(tmp_path / "probe")], capture_output=True, text=True, check=True).stdout.split("\n")
    for (c, f), line in zip(probes, lines):
        cls = getattr(_lib, c)
        assert line == f"{C.sizeof(cls)} {getattr(cls, f).offset}", (c, f)
