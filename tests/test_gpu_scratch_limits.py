"""Workspaces sized for a longer call (C ABI): a shorter call, whose own plan may want more room, runs in them, at the limit to
the byte, with the results of a workspace of its own size."""
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


def _dims(a, lens, HQ, H, D):
    T = sum(lens)
    a.T_tot, a.N, a.NT, a.HQ, a.H, a.K, a.V, a.M = T, len(lens), sum((n + 63) // 64 for n in lens), HQ, H, D, D, 64
    a.wl, a.shift, a.dtype, a.scale = 100, 0, _lib.NHA_DTYPE_BF16, D ** -0.5
    return a


def _smaller_workspace(cls, query, T, HQ, H, D):
    """Bytes that a longer call asks for, fewer than the call of T tokens does; None if there is no such call."""
    own = query(C.byref(_dims(cls(), [T], HQ, H, D)))
    sizes = [query(C.byref(_dims(cls(), [t], HQ, H, D))) for t in range(T + 64, 20 * T, 64)]
    least = min(sizes)
    return (own, least) if least < own else (own, None)


@pytest.mark.parametrize("T,HQ,H,D", [(1000, 8, 8, 128), (1152, 8, 8, 128), (1216, 16, 4, 64), (1088, 4, 4, 256), (2048, 8, 2, 128), (2048, 8, 2, 256)])
def test_forward_and_backward_in_a_longer_calls_workspace(T, HQ, H, D):
    lib = _lib.load()
    dev = torch.device("cuda:0")
    cu_d, idx_d, off_d, NT = prefill_tables(np.array([0, T], dtype=np.int32), dev)
    d = prefill_inputs(T, 1, T, HQ, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5, with_state=True)
    x = [d[k][0].contiguous().to(dev) for k in KEYS]
    h0 = [t.to(dev) for t in d["h0"]]
    new = lambda *s, dt=BF: torch.full(s, float("nan"), dtype=dt, device=dev)
    tight = 0
    own, small = _smaller_workspace(_lib.NhaPrefillArgs, lib.nha_prefill_scratch_bytes, T, HQ, H, D)
    outs = {}
    for size in filter(None, (own, small)):
        o, ls, lg = new(T, HQ, D), new(T, HQ, dt=torch.float32), new(T, HQ, dt=torch.float32)
        hk, hv = new(1, H, D, 64, dt=torch.float32), new(1, H, 64, D, dt=torch.float32)
        ws = torch.full((size + 256,), 255, dtype=torch.uint8, device=dev)
        a = _dims(_lib.NhaPrefillArgs(), [T], HQ, H, D)
        a.q_swa, a.k_swa, a.q_gsa, a.k_gsa, a.v, a.s, a.g = map(_ptr, x)
        a.o, a.lse_swa, a.lse_gsa, a.hkt, a.hvt, a.h0k, a.h0v = map(_ptr, (o, ls, lg, hk, hv, *h0))
        a.cu_seqlens, a.chunk_indices, a.chunk_offsets = map(_ptr, (cu_d, idx_d, off_d))
        a.scratch, a.scratch_bytes, a.stream = _ptr(ws), size, torch.cuda.current_stream().cuda_stream
        assert lib.nha_prefill_fwd(C.byref(a)) == 0, lib.nha_last_error()
        torch.cuda.synchronize()
        assert (ws[size:] == 255).all()
        outs[size] = (o, ls, lg, hk, hv)
        tight += size != own
    if small:      # longer segments keep fewer fp32 states: chunk-start states summed in another order and rounded to bf16 once
        for p, q in zip(outs[own], outs[small]):
            assert ((p.double() - q.double()).norm() / p.double().norm()).item() <= 5e-3
    o, ls, lg = outs[own][:3]
    do = torch.randn(T, HQ, D, generator=torch.Generator().manual_seed(1)).to(BF).to(dev)
    own, small = _smaller_workspace(_lib.NhaPrefillBwdArgs, lib.nha_prefill_bwd_scratch_bytes, T, HQ, H, D)
    grads = {}
    for size in filter(None, (own, small)):
        g = [torch.full_like(t, float("nan")) for t in x]
        ws = torch.full((size + 256,), 255, dtype=torch.uint8, device=dev)
        b = _dims(_lib.NhaPrefillBwdArgs(), [T], HQ, H, D)
        b.q_swa, b.k_swa, b.q_gsa, b.k_gsa, b.v, b.s, b.g = map(_ptr, x)
        b.o, b.lse_swa, b.lse_gsa, b.dout, b.h0k, b.h0v = map(_ptr, (o, ls, lg, do, *h0))
        b.dq_swa, b.dk_swa, b.dq_gsa, b.dk_gsa, b.dv, b.ds, b.dg = map(_ptr, g)
        b.cu_seqlens, b.chunk_indices, b.chunk_offsets = map(_ptr, (cu_d, idx_d, off_d))
        b.scratch, b.scratch_bytes, b.stream = _ptr(ws), size, torch.cuda.current_stream().cuda_stream
        assert lib.nha_prefill_bwd(C.byref(b)) == 0, lib.nha_last_error()
        torch.cuda.synchronize()
        assert (ws[size:] == 255).all() and all(t.isfinite().all() for t in g)
        grads[size] = g
        tight += size != own
    if small:
        for p, q in zip(grads[own], grads[small]):
            assert ((p.double() - q.double()).norm() / p.double().norm()).item() <= 1e-2
    assert tight, "no longer call with a smaller workspace: other sizes are needed here"


def test_too_small_is_refused():
    lib = _lib.load()
    x = torch.zeros(1 << 16, dtype=torch.uint8, device="cuda")
    a = _dims(_lib.NhaPrefillArgs(), [1000], 8, 8, 128)
    for f in ("q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g", "o", "cu_seqlens", "chunk_indices", "chunk_offsets", "scratch"):
        setattr(a, f, x.data_ptr())
    a.scratch_bytes = 1 << 16
    assert lib.nha_prefill_fwd(C.byref(a)) == _lib.NHA_ERR_SCRATCH
