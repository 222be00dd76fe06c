"""Head size 256 forward: sequences of an odd number of chunks, whose last workgroup has no second chunk, with window scores far
above the softmax reference.  Nothing outside the call's workspace is written, results are those of the fp32-math kernels, and a
sequence's bits do not depend on the one packed before it."""
import ctypes as C

import numpy as np
import pytest
import torch

from nha_amd import _lib
from nha_amd.ops import _ptr, prefill_tables
from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu
KEYS = ("q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g")
BF = torch.bfloat16
D = 256


@pytest.mark.parametrize("lens", [(40,), (64,), (150,), (192,), (64, 192, 40), (150, 100, 64)])
@pytest.mark.parametrize("wl", [99, -1])
def test_large_scores_stay_inside_the_workspace(lens, wl):
    """16 heads: the flags of the exact pass end where the workspace does, with no padding behind them."""
    from nha_amd import chunk_nha
    print("case", lens, wl, flush=True)
    lib, dev, H, T = _lib.load(), torch.device("cuda:0"), 16, sum(lens)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    cu_d, idx_d, off_d, NT = prefill_tables(cu, dev)
    d = prefill_inputs(T, 1, T, H, H, D, D, 64, dtype=BF, qk_scale=3.0)
    x = [d[k][0].contiguous().to(dev) for k in KEYS]
    o, ls, lg = (torch.full((T, H, *s), float("nan"), dtype=dt, device=dev) for s, dt in (((D,), BF), ((), torch.float32), ((), torch.float32)))
    a = _lib.NhaPrefillArgs()
    a.q_swa, a.k_swa, a.q_gsa, a.k_gsa, a.v, a.s, a.g = map(_ptr, x)
    a.o, a.lse_swa, a.lse_gsa, a.cu_seqlens, a.chunk_indices, a.chunk_offsets = map(_ptr, (o, ls, lg, cu_d, idx_d, off_d))
    a.T_tot, a.N, a.NT, a.HQ, a.H, a.K, a.V, a.M = T, len(lens), NT, H, H, D, D, 64
    a.wl, a.shift, a.dtype, a.impl, a.scale = wl, 0, _lib.NHA_DTYPE_BF16, _lib.NHA_IMPL_MFMA, 1.0
    size = lib.nha_prefill_scratch_bytes(C.byref(a))
    assert NT * H * 16 % 256 == 0
    ws = torch.zeros(size + 4096, dtype=torch.uint8, device=dev)      # zeros: a flag is a bit set
    a.scratch, a.scratch_bytes, a.stream = _ptr(ws), size, torch.cuda.current_stream().cuda_stream
    assert lib.nha_prefill_fwd(C.byref(a)) == 0, lib.nha_last_error()
    torch.cuda.synchronize()
    assert not ws[size:].any()
    want = chunk_nha(*(t[None] for t in x), cu_seqlens=cu_d, scale=1.0, window_size_left=wl, gsa_kv_shift=0, impl="simple")
    for name, got, ref in zip(("o", "lse_swa", "lse_gsa"), (o, ls, lg), want):      # bound: see test_gpu_prefill_mfma.py
        assert got.isfinite().all(), name
        assert ((got.double() - ref[0].double()).norm() / ref.double().norm()).item() <= 3e-2, name


@pytest.mark.parametrize("n", [40, 64, 150, 192, 200])
@pytest.mark.parametrize("after", [30, 100])
def test_a_sequence_keeps_its_bits_behind_any_other(n, after):
    from nha_amd import chunk_nha
    print("case", n, after, flush=True)
    H = 4
    d = prefill_inputs(n + after, 1, n + after, H, H, D, D, 64, dtype=BF, qk_scale=0.05)
    cu = torch.tensor([0, n, n + after], dtype=torch.int32, device="cuda")
    outs = []
    for factor in (1.0, 60.0):
        x = [d[k].clone() for k in KEYS]
        for t in x[:2]:
            t[:, :n] *= factor
        outs.append(chunk_nha(*(t.cuda() for t in x), cu_seqlens=cu, scale=1.0, window_size_left=63, gsa_kv_shift=64, impl="mfma"))
    assert not torch.equal(outs[0][0][:, :n], outs[1][0][:, :n])
    for p, q in zip(*outs):
        assert torch.equal(p[:, n:], q[:, n:])
