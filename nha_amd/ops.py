"""Host-side mirror of the reference op API for the NHA hot path, bound to libnha_hip.so.

Same names, argument meaning, return tuples and error behaviour as
  nha_fla/ops/nha/chunk.py:568-690            chunk_nha
  nha_fla/ops/nha/chunk_fused.py:291-380      fused_chunk_nha_prefill
  nha_fla/ops/nha/fused_recurrent.py:431-584  fused_recurrent_nha_decode
  nha_fla/ops/nha/fused_recurrent.py:588-682  fused_recurrent_nha
Differences, all widening: k/v/s/g may carry fewer (kv) heads than q in chunk_nha (the reference
needs them pre-expanded); window and head-dim limits of the fused prefill are lifted.  chunk_nha
is differentiable (nha_prefill_bwd behind nha_fla/ops/nha/chunk.py:490-564); the inference ops
reject inputs that require grad, as the reference's do.
PyTorch is used for device memory and the current stream only; every tensor op on the hot path
is a HIP kernel behind the C ABI.  There is no CPU / eager fallback.
"""
from __future__ import annotations

import ctypes as C
import functools
import threading
import weakref
from typing import Optional, Tuple

import numpy as np
import torch

from . import _lib
from .varlen import CHUNK, chunk_tables

__all__ = ["chunk_nha", "fused_chunk_nha_prefill", "fused_recurrent_nha", "fused_recurrent_nha_decode",
           "prefill_tables", "nha_prefill", "nha_prefill_bwd", "nha_layer_prologue", "nha_layer_epilogue"]

_DT = {torch.float32: _lib.NHA_DTYPE_F32, torch.bfloat16: _lib.NHA_DTYPE_BF16}
_IMPL = {None: _lib.NHA_IMPL_AUTO, "auto": _lib.NHA_IMPL_AUTO, "simple": _lib.NHA_IMPL_SIMPLE,
         "mfma": _lib.NHA_IMPL_MFMA}


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _stream(dev) -> int:
    return torch._C._cuda_getCurrentRawStream(dev.index)      # a tensor's device: its index is never None


def _as(x: Optional[torch.Tensor], dt) -> Optional[torch.Tensor]:
    """x contiguous in dtype dt; x itself where it is that already (two attribute reads instead of two dispatched calls)."""
    return x if x is None or (x.dtype == dt and x.is_contiguous()) else x.to(dt).contiguous()


def _dtype_code(t: torch.Tensor) -> int:
    if t.dtype not in _DT:
        raise TypeError(f"NHA HIP kernels take bfloat16 or float32 tensors, got {t.dtype}")
    return _DT[t.dtype]


def _need_cuda(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise RuntimeError("NHA ops run on the GPU only (tensor on %s); there is no CPU fallback" % t.device)


# ---------------------------------------------------------------------------------------------
# varlen tables, cached per cu_seqlens content
# ---------------------------------------------------------------------------------------------
_TABLE_CACHE: dict = {}


def prefill_tables(cu_host: np.ndarray, device) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, int]:
    """(cu_seqlens, chunk_indices [NT,2], chunk_offsets [N+1]) as int32 device tensors + NT."""
    key = (cu_host.tobytes(), str(device))
    hit = _TABLE_CACHE.get(key)
    if hit is not None:
        return hit
    idx, off = chunk_tables(cu_host, CHUNK)
    out = (torch.from_numpy(cu_host.astype(np.int32)).to(device), torch.from_numpy(idx).to(device),
           torch.from_numpy(off).to(device), int(idx.shape[0]))
    if len(_TABLE_CACHE) > 64:
        _TABLE_CACHE.pop(next(iter(_TABLE_CACHE)))      # oldest entry
    _TABLE_CACHE[key] = out
    return out


# ---------------------------------------------------------------------------------------------
# forward workspace: one buffer per (device, stream), grown when a call needs more.  Calls on one
# stream are ordered by the stream, so they can share it; another stream gets its own.
# ---------------------------------------------------------------------------------------------
_WORKSPACE: dict = {}
_WORKSPACE_MAX_STREAMS = 16      # entries kept; the one used longest ago leaves first (streams come and go)


_POOL_LOCK = threading.Lock()    # of both pools: several threads take, evict and release (autograd's backward thread is one)


def _workspace(nbytes: int, dev, stream: int) -> torch.Tensor:
    key = (str(dev), stream)
    with _POOL_LOCK:
        ws = _WORKSPACE.pop(key, None)
        if ws is None or ws.numel() < nbytes:
            ws = torch.empty(max(nbytes, 1 << 20), dtype=torch.uint8, device=dev)
        _WORKSPACE[key] = ws             # re-inserted: the dict's order is the order of last use
        while len(_WORKSPACE) > _WORKSPACE_MAX_STREAMS:
            _WORKSPACE.pop(next(iter(_WORKSPACE)))
    return ws


# scratch of the decode steps (arrival counters, partial results): one small buffer per (device, stream), zero when it is
# made; a step leaves its counters zero again, so it serves every decode call of the stream
_DECODE_SCRATCH: dict = {}


def new_decode_scratch(dev) -> torch.Tensor:
    return torch.zeros(_lib.load().nha_decode_scratch_bytes(), dtype=torch.uint8, device=dev)


def decode_scratch(dev, stream: int) -> Optional[torch.Tensor]:
    if torch.cuda.is_current_stream_capturing():       # a recording keeps its own (run_decode)
        return None
    ws = _DECODE_SCRATCH.get((dev, stream))
    if ws is None:
        ws = new_decode_scratch(dev)
        with _POOL_LOCK:                               # threads with new streams of their own
            while len(_DECODE_SCRATCH) >= _WORKSPACE_MAX_STREAMS:
                _DECODE_SCRATCH.pop(next(iter(_DECODE_SCRATCH)))
            _DECODE_SCRATCH[(dev, stream)] = ws
    return ws


def run_decode(args: bytes, dev, scratch: Optional[torch.Tensor]) -> None:
    """The step of an argument block from pack_decode.  Without scratch (in a recording) one is made, zeroed at every replay,
    if the call needs it: the fill takes a replay 1.5 to 3 us."""
    lib = _lib.load()
    if scratch is None and lib.decode_uses_scratch_packed(args):
        scratch = new_decode_scratch(dev)
        args = _lib.with_scratch(args, scratch.data_ptr(), scratch.numel())
    rc = lib.decode_step_packed(args)
    if rc:
        _lib.check(rc)


def release_workspaces() -> int:
    """Drop the cached workspaces (prefill forward and backward, decode scratch) of every device and stream and return
    the bytes they held.  The buffers are grow-only: one large prefill otherwise keeps its scratch for the life of the
    process, out of reach of `torch.cuda.empty_cache()`.  Work already queued keeps its buffer alive through the
    caching allocator's stream ordering, so this is safe to call between steps."""
    with _POOL_LOCK:
        held = sum(ws.numel() for pool in (_WORKSPACE, _DECODE_SCRATCH) for ws in pool.values())
        _WORKSPACE.clear()
        _DECODE_SCRATCH.clear()
    return held


# host copies of cu_seqlens tensors, keyed by the tensor OBJECT (weakly) and its version counter, so that
# the layers of a model, which all receive the same tensor, wait for one device-to-host copy, not one each
_CU_HOST: dict = {}      # id(tensor) -> (weak reference, version, host copy)


def _cu_to_host(cu: torch.Tensor) -> np.ndarray:
    if not cu.is_cuda:
        return cu.detach().to(torch.int32).numpy()
    key = id(cu)
    hit = _CU_HOST.get(key)
    if hit is not None and hit[0]() is cu and hit[1] == cu._version:
        return hit[2]
    host = cu.detach().to("cpu", torch.int32).numpy()
    _CU_HOST[key] = (weakref.ref(cu, lambda _, k=key: _CU_HOST.pop(k, None)), cu._version, host)
    return host


def _token_major(q, k):
    """The packed entries number tokens by the first of three sizes; with another number of them the results would be
    allocated for other tokens than the kernels write."""
    if q.dim() != 3 or k.dim() != 3:
        raise ValueError(f"expected token-major tensors [T, heads, dim], got q_swa {tuple(q.shape)}, k_swa {tuple(k.shape)}")


def nha_prefill(q_swa, k_swa, q_gsa, k_gsa, v, s, g, cu_host: np.ndarray, *, wl: int, shift: int, scale: float,
                h0=None, want_state: bool = False, want_lse: bool = True, impl=None):
    """Packed prefill on token-major tensors ``[T_tot, heads, dim]`` (one nha_prefill_fwd call).
    Returns (o, lse_swa, lse_gsa, hkt, hvt)."""
    _token_major(q_swa, k_swa)
    return _prefill((q_swa, k_swa, q_gsa, k_gsa, v, s, g), q_swa.shape[:1], cu_host, wl, shift, scale, h0, want_state, want_lse, impl)


def _at(t: Optional[torch.Tensor]) -> int:
    return 0 if t is None else t.data_ptr()


def _prefill(args, lead, cu_host: np.ndarray, wl: int, shift: int, scale: float, h0, want_state: bool, want_lse: bool, impl):
    """nha_prefill on contiguous tensors ``[..., heads, dim]`` whose leading sizes number the same tokens; o and the
    logsumexps come back with the leading sizes `lead`.  Small calls are bound by this function: with the argument block
    packed (not 35 ctypes fields set) and no views made of operands and results, chunk_nha on 512 tokens of 4 fp32 heads of 64
    takes 34 us where it took 44, the host's share of it 31 where it was 47."""
    lib = _lib.load()
    q_swa, k_swa, v, s = args[0], args[1], args[4], args[5]
    HQ, K = q_swa.shape[-2:]
    T_tot = q_swa.shape[0] if q_swa.dim() == 3 else q_swa.shape[0] * q_swa.shape[1]
    H, V, M = k_swa.shape[-2], v.shape[-1], s.shape[-1]
    dev, dt = q_swa.device, q_swa.dtype
    N = cu_host.size - 1
    cu_d, idx_d, off_d, NT = prefill_tables(cu_host, dev)
    o = torch.empty(*lead, HQ, V, dtype=dt, device=dev)
    lse_swa = torch.empty(*lead, HQ, dtype=torch.float32, device=dev) if want_lse else None
    lse_gsa = torch.empty(*lead, HQ, dtype=torch.float32, device=dev) if want_lse else None
    hkt = torch.empty(N, H, K, M, dtype=torch.float32, device=dev) if want_state else None
    hvt = torch.empty(N, H, M, V, dtype=torch.float32, device=dev) if want_state else None
    h0k = h0v = None
    if h0 is not None and h0[0] is not None:
        h0k, h0v = _as(h0[0], torch.float32), _as(h0[1], torch.float32)
        if tuple(h0k.shape) != (N, H, K, M) or tuple(h0v.shape) != (N, H, M, V):
            raise ValueError(f"initial_state must be ([{N},{H},{K},{M}], [{N},{H},{M},{V}]) (kv-head count), "
                             f"got {tuple(h0k.shape)} / {tuple(h0v.shape)}")
    stream = _stream(dev)
    head = (*(x.data_ptr() for x in args), o.data_ptr(), _at(lse_swa), _at(lse_gsa), _at(h0k), _at(h0v), _at(hkt), _at(hvt),
            cu_d.data_ptr(), idx_d.data_ptr(), off_d.data_ptr())
    dims = (T_tot, N, NT, HQ, H, K, V, M, _lib.i32(int(wl)), _lib.i32(int(shift)), _dtype_code(q_swa), _IMPL[impl],
            _lib.f32(float(scale)), stream)
    nbytes = lib.prefill_scratch_bytes_packed(_lib.pack_prefill(*head, 0, 0, *dims))
    if nbytes == 0:
        _lib.check(_lib.NHA_ERR_INVALID)
    scratch = _workspace(nbytes, dev, stream)
    _lib.check(lib.prefill_fwd_packed(_lib.pack_prefill(*head, scratch.data_ptr(), scratch.numel(), *dims)))
    return o, lse_swa, lse_gsa, hkt, hvt


def nha_prefill_bwd(q_swa, k_swa, q_gsa, k_gsa, v, s, g, o, lse_swa, lse_gsa, dout, cu_host: np.ndarray, *,
                    wl: int, shift: int, scale: float, h0=None, dlse_swa=None, dlse_gsa=None, dht=None,
                    want_dh0: bool = False):
    """Packed prefill backward on token-major tensors (one nha_prefill_bwd call).  Returns
    (dq_swa, dk_swa, dq_gsa, dk_gsa, dv, ds, dg, dh0k, dh0v) -- the last two None unless wanted."""
    _token_major(q_swa, k_swa)
    return _prefill_bwd((q_swa, k_swa, q_gsa, k_gsa, v, s, g), o, lse_swa, lse_gsa, dout, cu_host, wl, shift, scale, h0, dlse_swa,
                        dlse_gsa, dht, want_dh0)


def _prefill_bwd(args, o, lse_swa, lse_gsa, dout, cu_host: np.ndarray, wl: int, shift: int, scale: float, h0, dlse_swa, dlse_gsa,
                 dht, want_dh0: bool):
    """nha_prefill_bwd on contiguous tensors ``[..., heads, dim]`` whose leading sizes number the same tokens; a gradient has
    its tensor's shape."""
    lib = _lib.load()
    q_swa, k_swa, v, s = args[0], args[1], args[4], args[5]
    HQ, K = q_swa.shape[-2:]
    T_tot = q_swa.shape[0] if q_swa.dim() == 3 else q_swa.shape[0] * q_swa.shape[1]
    H, V, M = k_swa.shape[-2], v.shape[-1], s.shape[-1]
    dev = q_swa.device
    N = cu_host.size - 1
    cu_d, idx_d, off_d, NT = prefill_tables(cu_host, dev)
    f32 = lambda x: _as(x, torch.float32)
    h0k, h0v = (None, None) if h0 is None or h0[0] is None else (f32(h0[0]), f32(h0[1]))
    dhkt, dhvt = (None, None) if dht is None else dht
    if (dhkt is None) != (dhvt is None):      # one final state unused downstream: its cotangent is zero
        dhkt = torch.zeros(N, H, K, M, dtype=torch.float32, device=dev) if dhkt is None else dhkt
        dhvt = torch.zeros(N, H, M, V, dtype=torch.float32, device=dev) if dhvt is None else dhvt
    dhkt, dhvt, dlse_swa, dlse_gsa = f32(dhkt), f32(dhvt), f32(dlse_swa), f32(dlse_gsa)
    dout = _as(dout, q_swa.dtype)
    outs = [torch.empty_like(x) for x in args]
    dh0k = torch.empty(N, H, K, M, dtype=torch.float32, device=dev) if want_dh0 else None
    dh0v = torch.empty(N, H, M, V, dtype=torch.float32, device=dev) if want_dh0 else None
    stream = _stream(dev)
    head = (*(x.data_ptr() for x in args), o.data_ptr(), lse_swa.data_ptr(), lse_gsa.data_ptr(), _at(h0k), _at(h0v), dout.data_ptr(),
            _at(dlse_swa), _at(dlse_gsa), _at(dhkt), _at(dhvt), *(x.data_ptr() for x in outs), _at(dh0k), _at(dh0v),
            cu_d.data_ptr(), idx_d.data_ptr(), off_d.data_ptr())
    dims = (T_tot, N, NT, HQ, H, K, V, M, _lib.i32(int(wl)), _lib.i32(int(shift)), _dtype_code(q_swa), _lib.f32(float(scale)), stream)
    nbytes = lib.prefill_bwd_scratch_bytes_packed(_lib.pack_prefill_bwd(*head, 0, 0, *dims))
    if nbytes == 0:
        _lib.check(_lib.NHA_ERR_INVALID)
    scratch = _workspace(nbytes, dev, stream)     # shared with the forward: calls on one stream are ordered
    _lib.check(lib.prefill_bwd_packed(_lib.pack_prefill_bwd(*head, scratch.data_ptr(), nbytes, *dims)))
    return (*outs, dh0k, dh0v)


class _Refusal(torch.autograd.Function):
    """The first n of the tensors, as functions of the others that have no derivative."""

    @staticmethod
    def forward(ctx, n, *tensors):
        return tuple(t.detach() for t in tensors[:n])

    @staticmethod
    def backward(ctx, *grads):
        raise RuntimeError("the NHA kernels have first derivatives only: this gradient cannot be differentiated twice")


class _SavedOnce:
    """A node's context whose saved tensors are unpacked once (torch.utils.checkpoint gives them out once)."""

    def __init__(self, ctx):
        self._ctx, self.saved_tensors = ctx, ctx.saved_tensors

    def __getattr__(self, name):
        return getattr(self._ctx, name)


def _first_derivatives_only(backward):
    """For an autograd node whose backward is a kernel.  Under create_graph its gradients hang on everything that they were
    formed from, through a node that raises: a second derivative that passes through here is refused, also one that reaches
    its input by another way too (a residual connection), where torch's once_differentiable, whose node hangs on nothing, is
    passed by and the sum comes out without the terms of this node."""
    @functools.wraps(backward)
    def wrapped(ctx, *grads):
        if not torch.is_grad_enabled():
            return backward(ctx, *grads)
        ctx = _SavedOnce(ctx)
        with torch.no_grad():
            outs = backward(ctx, *grads)
        roots = [t for t in (*grads, *ctx.saved_tensors) if t is not None and t.requires_grad]
        formed = [t for t in outs if t is not None]
        if roots and formed:
            new = iter(_Refusal.apply(len(formed), *formed, *roots))
            outs = tuple(None if t is None else next(new) for t in outs)
        return outs
    return wrapped


_FMAP = {None: _lib.NHA_FMAP_NONE, "none": _lib.NHA_FMAP_NONE, "swish": _lib.NHA_FMAP_SWISH, "relu": _lib.NHA_FMAP_RELU}


def _prologue_dims(q, k, v, f, inv_freq, cu):
    B, T, HQ, K = q.shape
    H, V, M = k.shape[2], v.shape[3], f.shape[3]
    if cu is not None and B != 1:
        raise ValueError("cu_seqlens needs the packed layout [1, T_tot, ...]")
    for x in (k, v, f):
        if x.dtype != q.dtype:
            raise TypeError("q, k, v, f must share one dtype")
    if inv_freq.numel() != K // 2:
        raise ValueError(f"inv_freq must hold K/2 = {K // 2} entries, got {inv_freq.numel()}")
    return dict(T_tot=B * T, N=(cu.numel() - 1) if cu is not None else B, HQ=HQ, H=H, K=K, V=V, M=M)


def _prologue_fwd(q, k, v, f, inv_freq, fm: int, normalizer: float, offset: int, cu):
    lib = _lib.load()
    dims = _prologue_dims(q, k, v, f, inv_freq, cu)
    q_swa, k_swa, v_out = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    s, g = torch.empty_like(f), torch.empty_like(f)
    q_gsa = torch.empty_like(q) if fm else None
    k_gsa = torch.empty_like(k) if fm else None
    a = _lib.NhaLayerPrologueArgs(
        q=_ptr(q), k=_ptr(k), v=_ptr(v), f=_ptr(f), q_swa=_ptr(q_swa), k_swa=_ptr(k_swa), q_gsa=_ptr(q_gsa),
        k_gsa=_ptr(k_gsa), v_out=_ptr(v_out), s=_ptr(s), g=_ptr(g), inv_freq=_ptr(inv_freq), cu_seqlens=_ptr(cu),
        feature_map=fm, seqlen_offset=int(offset), dtype=_dtype_code(q), gate_logit_normalizer=float(normalizer),
        stream=_stream(q.device), **dims)
    _lib.check(lib.nha_layer_prologue(C.byref(a)))
    return q_swa, k_swa, q_gsa, k_gsa, v_out, s, g


def _prologue_bwd(q, k, v, f, inv_freq, fm: int, normalizer: float, offset: int, cu, dq_swa, dk_swa, dq_gsa, dk_gsa,
                  dv_out, ds, dg):
    lib = _lib.load()
    dims = _prologue_dims(q, k, v, f, inv_freq, cu)
    dq, dk, dv, df = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), torch.empty_like(f)
    a = _lib.NhaLayerPrologueBwdArgs(
        q=_ptr(q), k=_ptr(k), v=_ptr(v), f=_ptr(f), dq_swa=_ptr(dq_swa), dk_swa=_ptr(dk_swa), dq_gsa=_ptr(dq_gsa),
        dk_gsa=_ptr(dk_gsa), dv_out=_ptr(dv_out), ds=_ptr(ds), dg=_ptr(dg), dq=_ptr(dq), dk=_ptr(dk), dv=_ptr(dv),
        df=_ptr(df), inv_freq=_ptr(inv_freq), cu_seqlens=_ptr(cu), feature_map=fm, seqlen_offset=int(offset),
        dtype=_dtype_code(q), gate_logit_normalizer=float(normalizer), stream=_stream(q.device), **dims)
    _lib.check(lib.nha_layer_prologue_bwd(C.byref(a)))
    return dq, dk, dv, df


class _LayerPrologueFunction(torch.autograd.Function):
    """Autograd node of the fused prologue: both directions are one HIP launch."""

    @staticmethod
    def forward(ctx, q, k, v, f, inv_freq, fm, normalizer, offset, cu):
        outs = _prologue_fwd(q, k, v, f, inv_freq, fm, normalizer, offset, cu)
        ctx.save_for_backward(q, k, v, f, inv_freq)
        ctx.cu, ctx.meta = cu, (fm, normalizer, offset)
        return outs if fm else (outs[0], outs[1], outs[4], outs[5], outs[6])

    @staticmethod
    @_first_derivatives_only
    def backward(ctx, *grads):
        q, k, v, f, inv_freq = ctx.saved_tensors
        fm, normalizer, offset = ctx.meta
        shapes = (q, k, q, k, v, f, f) if fm else (q, k, v, f, f)
        grads = [torch.zeros_like(x) if gr is None else gr.contiguous() for gr, x in zip(grads, shapes)]
        if fm:
            dq_swa, dk_swa, dq_gsa, dk_gsa, dv_out, ds, dg = grads
        else:
            (dq_swa, dk_swa, dv_out, ds, dg), dq_gsa, dk_gsa = grads, None, None
        dq, dk, dv, df = _prologue_bwd(q, k, v, f, inv_freq, fm, normalizer, offset, ctx.cu, dq_swa, dk_swa, dq_gsa,
                                       dk_gsa, dv_out, ds, dg)
        return dq, dk, dv, df, None, None, None, None, None


def nha_layer_prologue(q, k, v, f, inv_freq, *, feature_map: Optional[str], gate_logit_normalizer: float,
                       seqlen_offset: int = 0, cu_seqlens: Optional[torch.Tensor] = None, projections=None):
    """One launch for the elementwise chain of nha_fla/layers/nha.py:214-237 on the raw projections
    q [B,T,HQ,K], k [B,T,H,K], v [B,T,H,V], f [B,T,H,M] (B = 1 with cu_seqlens, an int32 device
    tensor).  Returns (q_swa, k_swa, q_gsa, k_gsa, v, s, g); without a feature map q_gsa / k_gsa
    are q / k themselves.  Differentiable with respect to q, k, v, f (one launch backward too).

    projections: (x [B,T,hidden], the q, k, v, f projection modules, (HQ, H, K, V, M)) in the place of q, k, v, f: one autograd
    node with the projections (_layer_front) where layer_front_supported accepts them and there is a feature map, the modules'
    own outputs elsewhere."""
    if feature_map not in _FMAP:
        raise NotImplementedError(f"Feature map `{feature_map}` has no fused prologue.")
    if projections is not None:
        x, modules, (HQ, H, K, V, M) = projections
        if _FMAP[feature_map] and (isinstance(projections, _FrontProjections) or layer_front_supported(*projections)):
            return _layer_front(x, modules, (HQ, H, K, V, M), inv_freq, feature_map=feature_map,
                                gate_logit_normalizer=gate_logit_normalizer, seqlen_offset=seqlen_offset, cu_seqlens=cu_seqlens)
        q, k, v, f = (y.unflatten(-1, d) for y, d in zip(shared_input_linears(x, modules), ((HQ, K), (H, K), (H, V), (H, M))))
    _need_cuda(q, k, v, f, inv_freq, cu_seqlens)
    _dtype_code(q)
    q, k, v, f = (x.contiguous() for x in (q, k, v, f))
    inv_freq = inv_freq.detach().to(torch.float32).contiguous()
    fm = _FMAP[feature_map]
    cu = None if cu_seqlens is None else cu_seqlens.to(device=q.device, dtype=torch.int32).contiguous()
    args = (q, k, v, f, inv_freq, fm, float(gate_logit_normalizer), int(seqlen_offset), cu)
    if torch.is_grad_enabled() and any(x.requires_grad for x in (q, k, v, f)):
        outs = _LayerPrologueFunction.apply(*args)
        if fm:
            return outs
        return outs[0], outs[1], q, k, outs[2], outs[3], outs[4]
    q_swa, k_swa, q_gsa, k_gsa, v_out, s, g = _prologue_fwd(*args)
    return q_swa, k_swa, (q_gsa if fm else q), (k_gsa if fm else k), v_out, s, g


def _layer_front(x, modules, dims, inv_freq, *, feature_map: str, gate_logit_normalizer: float, seqlen_offset: int = 0,
                 cu_seqlens: Optional[torch.Tensor] = None):
    """nha_layer_prologue on the outputs of the q, k, v, f projection `modules` of x [B,T,hidden], projections and prologue as
    one node; for calls that layer_front_supported accepts.  dims: (HQ, H, K, V, M).  The weights side by side are one product
    instead of four, and one for the input's gradient: layer step of 1400 tokens (host-bound) 1010 -> 865 us, of 16384
    tokens 1778 -> 1731."""
    if cu_seqlens is not None and x.shape[0] != 1:
        raise ValueError("cu_seqlens needs the packed layout [1, T_tot, ...]")
    if inv_freq.numel() != dims[2] // 2 or inv_freq.device != x.device:
        raise ValueError(f"inv_freq must hold K/2 = {dims[2] // 2} entries on {x.device}, got {inv_freq.numel()} on {inv_freq.device}")
    cu = None if cu_seqlens is None else cu_seqlens.to(device=x.device, dtype=torch.int32).contiguous()
    return _LayerFrontFunction.apply(x, *(m.weight for m in modules), inv_freq.detach().to(torch.float32).contiguous(),
                                     tuple(dims), _FMAP[feature_map], float(gate_logit_normalizer), int(seqlen_offset), cu)


def _epilogue_fwd(o, w, b, eps: float):
    lib = _lib.load()
    dim = o.shape[-1]
    y = torch.empty_like(o)
    a = _lib.NhaLayerEpilogueArgs(o=_ptr(o), y=_ptr(y), weight=_ptr(w), bias=_ptr(b), rows=o.numel() // dim, dim=dim,
                                  dtype=_dtype_code(o), eps=float(eps), stream=_stream(o.device))
    _lib.check(lib.nha_layer_epilogue(C.byref(a)))
    return y


class _LayerEpilogueFunction(torch.autograd.Function):
    """Autograd node of the fused epilogue; the weight / bias gradients are reduced from the
    kernel's per-workgroup partial sums in a fixed order."""

    @staticmethod
    def forward(ctx, o, weight, bias, eps):
        w = None if weight is None else weight.detach().to(torch.float32).contiguous()
        b = None if bias is None else bias.detach().to(torch.float32).contiguous()
        ctx.save_for_backward(o, w)
        ctx.eps = eps
        ctx.wb = (None if weight is None else weight.dtype, None if bias is None else bias.dtype)
        return _epilogue_fwd(o, w, b, eps)

    @staticmethod
    @_first_derivatives_only
    def backward(ctx, dy):
        lib = _lib.load()
        o, w = ctx.saved_tensors
        dy = dy.contiguous()
        dim = o.shape[-1]
        rows = o.numel() // dim
        parts = lib.nha_layer_epilogue_bwd_parts(rows)
        wdt, bdt = ctx.wb
        need_w = wdt is not None and ctx.needs_input_grad[1]
        need_b = bdt is not None and ctx.needs_input_grad[2]
        dwp = torch.empty(parts, dim, dtype=torch.float32, device=o.device) if need_w else None
        dbp = torch.empty(parts, dim, dtype=torch.float32, device=o.device) if need_b else None
        do = torch.empty_like(o)
        a = _lib.NhaLayerEpilogueBwdArgs(o=_ptr(o), dy=_ptr(dy), dout=_ptr(do), weight=_ptr(w), dweight_partial=_ptr(dwp),
                                         dbias_partial=_ptr(dbp), rows=rows, dim=dim, dtype=_dtype_code(o),
                                         eps=float(ctx.eps), stream=_stream(o.device))
        _lib.check(lib.nha_layer_epilogue_bwd(C.byref(a)))
        return (do, dwp.sum(0).to(wdt) if need_w else None, dbp.sum(0).to(bdt) if need_b else None, None)


def nha_layer_epilogue(o, weight: Optional[torch.Tensor], bias: Optional[torch.Tensor], eps: float):
    """rms_norm(silu(o)) * weight (+ bias) over the last dimension in one launch: the normalisation
    half of nha_fla/layers/nha.py:278.  Differentiable with respect to o, weight and bias (last
    dimension a multiple of 8 and at most 8192 for the backward)."""
    _need_cuda(o, weight, bias)
    _dtype_code(o)
    o = o.contiguous()
    if torch.is_grad_enabled() and any(x is not None and x.requires_grad for x in (o, weight, bias)):
        dim = o.shape[-1]
        if dim % 8 or dim > 8192:
            raise NotImplementedError(f"nha_layer_epilogue backward needs a last dimension % 8 == 0 and <= 8192, got {dim}")
        return _LayerEpilogueFunction.apply(o, weight, bias, float(eps))
    w = None if weight is None else weight.detach().to(torch.float32).contiguous()
    b = None if bias is None else bias.detach().to(torch.float32).contiguous()
    return _epilogue_fwd(o, w, b, float(eps))


def nha_wgrad(x: torch.Tensor, dys) -> list:
    """dy^T x for every dy [T, O] of `dys` (at most four), x [T, I]: the weight gradients of projections of one input, bf16."""
    lib = _lib.load()
    if not 1 <= len(dys) <= 4 or x.dim() != 2 or any(dy.dim() != 2 or dy.shape[0] != x.shape[0] for dy in dys):
        raise ValueError(f"nha_wgrad takes x [T, I] and one to four dy [T, O], got {[tuple(t.shape) for t in (x, *dys)]}")
    if any(t.dtype != torch.bfloat16 or not t.is_cuda or t.device != x.device for t in (x, *dys)):
        raise TypeError("nha_wgrad takes bfloat16 tensors on one GPU")
    x = x.contiguous()
    T, width = x.shape
    # columns of one matrix are read where they are; rows that lie otherwise are made dense
    ldy = 0
    if not all(dy.is_contiguous() for dy in dys):
        ldy = dys[0].stride(0)
        if ldy % 8 or any(dy.stride() != (ldy, 1) or dy.shape[1] > ldy for dy in dys):
            dys, ldy = [dy.contiguous() for dy in dys], 0
    outs = [torch.empty(dy.shape[1], width, dtype=x.dtype, device=x.device) for dy in dys]
    a = _lib.NhaWgradArgs(x=_ptr(x), n=len(outs), T=T, I=width, ldy=ldy, stream=_stream(x.device))
    for i, (dy, dw) in enumerate(zip(dys, outs)):
        a.dy[i], a.dw[i], a.O[i] = _ptr(dy), _ptr(dw), dy.shape[1]
    nbytes = lib.nha_wgrad_scratch_bytes(C.byref(a))
    if nbytes == 0:
        _lib.check(_lib.NHA_ERR_INVALID)
    # of the call's own: it holds the partial sums between two launches, and another thread of this stream may queue a call that
    # uses the stream's shared workspace between them
    scratch = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    a.scratch, a.scratch_bytes = _ptr(scratch), nbytes
    _lib.check(lib.nha_wgrad(C.byref(a)))
    return outs


def _wgrad_supported(x: torch.Tensor, dys) -> bool:
    """Rows of 16-byte pieces, bf16, and sizes at which nha_wgrad is the faster one.  A single gradient of few tokens stays with
    the library: 1024 x 1024 from 4096 tokens takes it 30 us against 34, from 6000 45 against 39, from 16384 102 against 54;
    2048 x 2048 from 6000 72 against 67.  Several at once are faster from any number (1024 columns, outputs of 3 x 1024 + 512
    from 300 tokens: 28 us against 76 for four library calls).  Large weights are the library's, whose tiles of 256 columns fill
    the chip without a split there: a single 3072 x 3072 from 16384 tokens 303 us against 325; 3072 columns, 3072 + 2 x 768 + 512
    (15.7 M elements) from 1024 tokens 77 against 59, from 16384 703 against 488, but 4096 columns, 4096 + 2 x 1024 + 512 (27 M)
    80 against 100 and 916 against 902, and 3 x 4096 + 512 (52 M) 124 against 193 and 1512 against 1707."""
    T, width = x.shape
    elements = sum(dy.shape[1] for dy in dys) * width
    return (x.dtype == torch.bfloat16 and 0 < T <= 1 << 30 and width % 8 == 0 and x.data_ptr() % 16 == 0 and len(dys) <= 4
            and all(dy.dtype == x.dtype and dy.shape[1] % 8 == 0 and dy.data_ptr() % 16 == 0 for dy in dys)
            and (elements <= 1 << 24 if len(dys) > 1 else elements <= 1 << 22 and T >= 6000))


class _SharedInputLinear(torch.autograd.Function):
    """F.linear of one input with several weights.  Backward: the input's gradient summed inside the products (each added
    to the one before it, no tensors in between), the weights' gradients in one launch (nha_wgrad)."""

    @staticmethod
    def forward(ctx, x, *weights):
        ctx.save_for_backward(x, *weights)
        return tuple(torch.nn.functional.linear(x, w) for w in weights)

    @staticmethod
    def backward(ctx, *dys):
        x, *weights = ctx.saved_tensors
        rows = [dy.reshape(-1, dy.shape[-1]) for dy in dys]
        xr = x.reshape(-1, x.shape[-1])
        need = [i for i, n in enumerate(ctx.needs_input_grad[1:]) if n]
        dx, dws = None, [None] * len(weights)
        if torch.is_grad_enabled():                        # a second derivative is wanted: operations that have one
            if ctx.needs_input_grad[0]:
                dx = sum(dy @ w for dy, w in zip(rows, weights)).view(x.shape)
            for i in need:
                dws[i] = rows[i].t() @ xr
            return (dx, *dws)
        if ctx.needs_input_grad[0]:
            dx = rows[0] @ weights[0]
            for dy, w in zip(rows[1:], weights[1:]):
                dx.addmm_(dy, w)
            dx = dx.view(x.shape)
        picked, xc = [rows[i].contiguous() for i in need], xr.contiguous()
        if need and _wgrad_supported(xc, picked):
            for i, dw in zip(need, nha_wgrad(xc, picked)):
                dws[i] = dw
        else:
            for i in need:
                dws[i] = rows[i].t() @ xr
        return (dx, *dws)


class _LayerFrontFunction(torch.autograd.Function):
    """The four projections and the prologue of the layer as one node: one product with the weights side by side, whose
    columns the prologue reads where they are (nha_layer_prologue_rows); backward, the prologue's gradients side by side
    again, one product for the input's gradient and one launch for the weights'."""

    @staticmethod
    def forward(ctx, x, wq, wk, wv, wf, inv_freq, dims, fm, normalizer, offset, cu):
        HQ, H, K, V, M = dims
        B, T = x.shape[:2]
        raw = torch.nn.functional.linear(x, torch.cat([wq, wk, wv, wf]))
        new = lambda heads, width: torch.empty(B, T, heads, width, dtype=x.dtype, device=x.device)
        outs = (new(HQ, K), new(H, K), new(HQ, K), new(H, K), new(H, V), new(H, M), new(H, M))
        q_swa, k_swa, q_gsa, k_gsa, v, s, g = outs
        at = _front_columns(raw, dims)
        a = _lib.NhaLayerPrologueArgs(
            q=at[0], k=at[1], v=at[2], f=at[3], q_swa=_ptr(q_swa), k_swa=_ptr(k_swa), q_gsa=_ptr(q_gsa), k_gsa=_ptr(k_gsa),
            v_out=_ptr(v), s=_ptr(s), g=_ptr(g), inv_freq=_ptr(inv_freq), cu_seqlens=_ptr(cu), feature_map=fm,
            seqlen_offset=offset, dtype=_dtype_code(x), gate_logit_normalizer=normalizer, stream=_stream(x.device), T_tot=B * T,
            N=B if cu is None else cu.numel() - 1, HQ=HQ, H=H, K=K, V=V, M=M)
        _lib.check(_lib.load().nha_layer_prologue_rows(C.byref(a), raw.shape[-1]))
        ctx.save_for_backward(x, wq, wk, wv, wf, raw, inv_freq)
        ctx.cu, ctx.meta = cu, (dims, fm, normalizer, offset)
        return outs

    @staticmethod
    @_first_derivatives_only
    def backward(ctx, *grads):
        x, wq, wk, wv, wf, raw, inv_freq = ctx.saved_tensors
        (HQ, H, K, V, M), fm, normalizer, offset = ctx.meta
        B, T = x.shape[:2]
        grads = [gr.contiguous() for gr in grads]
        draw = torch.empty_like(raw)
        at, to = _front_columns(raw, ctx.meta[0]), _front_columns(draw, ctx.meta[0])
        dq_swa, dk_swa, dq_gsa, dk_gsa, dv, ds, dg = (_ptr(gr) for gr in grads)
        a = _lib.NhaLayerPrologueBwdArgs(
            q=at[0], k=at[1], v=at[2], f=at[3], dq_swa=dq_swa, dk_swa=dk_swa, dq_gsa=dq_gsa, dk_gsa=dk_gsa, dv_out=dv, ds=ds, dg=dg,
            dq=to[0], dk=to[1], dv=to[2], df=to[3], inv_freq=_ptr(inv_freq), cu_seqlens=_ptr(ctx.cu), feature_map=fm,
            seqlen_offset=offset, dtype=_dtype_code(x), gate_logit_normalizer=normalizer, stream=_stream(x.device), T_tot=B * T,
            N=B if ctx.cu is None else ctx.cu.numel() - 1, HQ=HQ, H=H, K=K, V=V, M=M)
        _lib.check(_lib.load().nha_layer_prologue_bwd_rows(C.byref(a), raw.shape[-1]))
        weights = (wq, wk, wv, wf)
        rows = draw.view(B * T, -1)
        dys = rows.split([w.shape[0] for w in weights], dim=1)
        xr = x.reshape(B * T, -1)
        dx, dws = None, [None] * 4
        if ctx.needs_input_grad[0]:
            dx = (rows @ torch.cat(weights)).view(x.shape)
        need = [i for i in range(4) if ctx.needs_input_grad[1 + i]]
        picked, xc = [dys[i] for i in need], xr.contiguous()
        if need and _wgrad_supported(xc, picked):
            for i, dw in zip(need, nha_wgrad(xc, picked)):
                dws[i] = dw
        else:
            for i in need:
                dws[i] = dys[i].t() @ xr
        return (dx, *dws, None, None, None, None, None, None)


def _front_columns(raw: torch.Tensor, dims):
    """Addresses of the q, k, v and f columns of the projections side by side."""
    HQ, H, K, V, M = dims
    p, size = raw.data_ptr(), raw.element_size()
    return p, p + HQ * K * size, p + (HQ + H) * K * size, p + ((HQ + H) * K + H * V) * size


_LINEAR_FORWARD = torch.nn.Linear.forward


def _for_one_node(x: torch.Tensor) -> bool:
    """Whether it is worth looking over the modules: not in inference (10 us of host time per layer call), nor where the look
    itself would be compiled."""
    return torch.is_grad_enabled() and not torch.compiler.is_compiling() and x.is_cuda and x.dtype == torch.bfloat16


def _one_node(x: torch.Tensor, weights) -> bool:
    """Whether a node of our own may stand for F.linear of x with every weight: something to differentiate, and nothing
    besides reverse-mode autograd that looks at the call (autocast, tracing, modes, transforms, subclasses)."""
    return (_for_one_node(x) and not torch.is_autocast_enabled("cuda")
            and all(w.dtype == x.dtype and w.device == x.device for w in weights)
            and any(t.requires_grad for t in (x, *weights)) and _plain_autograd((x, *weights)))


def _plain_modules(modules) -> bool:
    """nn.Linear modules without bias, hooks or a forward of their own."""
    return (torch.nn.Linear.forward is _LINEAR_FORWARD
            and not torch.nn.modules.module._has_any_global_hook()
            and all(type(m) is torch.nn.Linear and "forward" not in m.__dict__ and m.bias is None
                    and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks)
                    for m in modules))


def shared_input_linears(x: torch.Tensor, modules):
    """[m(x) for m in modules], as one autograd node where it may be one."""
    weights = [m.weight for m in modules] if _for_one_node(x) and _plain_modules(modules) else None
    if weights is not None and _one_node(x, weights):
        return _SharedInputLinear.apply(x, *weights)
    return tuple(m(x) for m in modules)


def layer_front_supported(x: torch.Tensor, modules, dims) -> bool:
    """Whether nha_layer_prologue takes (x, modules, dims) as its projections: plain modules whose products with x
    [B, T, hidden] and the prologue may be one autograd node.  dims: query heads, kv-heads, key size, value size, slots."""
    HQ, H, K, V, M = dims
    if not _for_one_node(x) or not _plain_modules(modules) or x.dim() != 3 or x.numel() == 0 or K % 2 or K > 1024:
        return False
    weights = [m.weight for m in modules]
    return (all(tuple(w.shape) == (n, x.shape[-1]) and n % 8 == 0 for w, n in zip(weights, (HQ * K, H * K, H * V, H * M)))
            and _one_node(x, weights))


class _FrontProjections(tuple):
    """(x, modules, dims) that layer_front_supported has accepted."""


def layer_front_projections(x: torch.Tensor, modules, dims) -> Optional[_FrontProjections]:
    """What the next nha_layer_prologue call takes as its projections without looking them over a second time, or None for
    what layer_front_supported refuses."""
    return _FrontProjections((x, modules, dims)) if layer_front_supported(x, modules, dims) else None


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    """F.linear, its weight gradient by nha_wgrad where that is the faster one."""
    if bias is None and _one_node(x, [weight]):
        return _SharedInputLinear.apply(x, weight)[0]
    return torch.nn.functional.linear(x, weight, bias)


@torch.compiler.disable
def gsa_share_begin(lse_swa: torch.Tensor, lse_gsa: torch.Tensor):
    """Starts forming the mean over tokens and heads of e^lse_gsa / (e^lse_swa + e^lse_gsa) (fp32 tensors of one shape) on
    the current stream: one launch and a copy of its partial sums to the host.  gsa_share_end waits for the value, so work
    queued between the two runs under the wait."""
    _need_cuda(lse_swa, lse_gsa)
    if lse_swa.dtype != torch.float32 or lse_gsa.dtype != torch.float32 or lse_swa.shape != lse_gsa.shape:
        raise ValueError("gsa_share takes two float32 tensors of one shape")
    a, b = lse_swa.detach().contiguous(), lse_gsa.detach().contiguous()
    n = a.numel()
    part = torch.empty(min(256, (n + 255) // 256), dtype=torch.float32, device=a.device)
    _lib.check(_lib.load().nha_gsa_share(a.data_ptr(), b.data_ptr(), n, part.data_ptr(), part.numel(), _stream(a.device)))
    host = torch.empty(part.numel(), dtype=torch.float32, pin_memory=True)
    host.copy_(part, non_blocking=True)
    done = torch.cuda.Event()
    done.record(torch.cuda.current_stream(a.device))
    return done, host, n


@torch.compiler.disable
def gsa_share_end(pending) -> float:
    done, host, n = pending
    done.synchronize()
    return sum(host.tolist()) / n


def gsa_share(lse_swa: torch.Tensor, lse_gsa: torch.Tensor) -> float:
    """Mean over tokens and heads of e^lse_gsa / (e^lse_swa + e^lse_gsa)."""
    return gsa_share_end(gsa_share_begin(lse_swa, lse_gsa))


def _short_conv_args(x, cu):
    T_tot = x.shape[0] * x.shape[1]
    N = (cu.numel() - 1) if cu is not None else x.shape[0]
    return T_tot, N


class _ShortConvFunction(torch.autograd.Function):
    """Autograd node of the short convolution: one launch per direction; the weight / bias gradients are
    reduced from the kernel's per-run partial sums in a fixed order."""

    @staticmethod
    def forward(ctx, x, weight, bias, cu, act):
        lib = _lib.load()
        Cn, KS = weight.shape[0], weight.shape[-1]
        w = weight.detach().to(x.dtype).reshape(Cn, KS).contiguous()
        b = None if bias is None else bias.detach().to(x.dtype).contiguous()
        T_tot, N = _short_conv_args(x, cu)
        y = torch.empty_like(x)
        a = _lib.NhaShortConvArgs(x=_ptr(x), weight=_ptr(w), bias=_ptr(b), y=_ptr(y), cu_seqlens=_ptr(cu), T_tot=T_tot, N=N,
                                  C=Cn, KS=KS, activation=int(act), dtype=_dtype_code(x), stream=_stream(x.device))
        _lib.check(lib.nha_short_conv(C.byref(a)))
        ctx.save_for_backward(x, w, b, cu)
        ctx.act = int(act)
        ctx.wb = (weight.dtype, weight.shape, None if bias is None else bias.dtype)
        return y

    @staticmethod
    @_first_derivatives_only
    def backward(ctx, dy):
        lib = _lib.load()
        x, w, b, cu = ctx.saved_tensors
        dy = dy.contiguous()
        Cn, KS = w.shape
        T_tot, N = _short_conv_args(x, cu)
        parts = lib.nha_short_conv_bwd_parts(T_tot)
        wdt, wshape, bdt = ctx.wb
        need_w = ctx.needs_input_grad[1]
        need_b = bdt is not None and ctx.needs_input_grad[2]
        dwp = torch.empty(parts, Cn, KS, dtype=torch.float32, device=x.device) if need_w else None
        dbp = torch.empty(parts, Cn, dtype=torch.float32, device=x.device) if need_b else None
        dx = torch.empty_like(x)
        a = _lib.NhaShortConvBwdArgs(x=_ptr(x), weight=_ptr(w), bias=_ptr(b), dy=_ptr(dy), dx=_ptr(dx), dweight_partial=_ptr(dwp),
                                     dbias_partial=_ptr(dbp), cu_seqlens=_ptr(cu), T_tot=T_tot, N=N, C=Cn, KS=KS,
                                     activation=ctx.act, dtype=_dtype_code(x), stream=_stream(x.device))
        _lib.check(lib.nha_short_conv_bwd(C.byref(a)))
        return (dx, dwp.sum(0).to(wdt).reshape(wshape) if need_w else None, dbp.sum(0).to(bdt) if need_b else None, None, None)


def short_conv_supported(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether nha_short_conv serves this call: GPU tensors in bf16 / fp32, 2 to 4 taps, channels a multiple of 8."""
    return (x.is_cuda and x.dtype in (torch.bfloat16, torch.float32) and 2 <= weight.shape[-1] <= 4
            and weight.shape[0] % 8 == 0)


def nha_short_conv(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], *,
                   cu_seqlens: Optional[torch.Tensor] = None, activation: Optional[str] = "silu") -> torch.Tensor:
    """Depthwise causal convolution over ``x [B, T, C]`` with ``weight [C, 1, KS]`` (+ ``bias [C]``) and optional
    SiLU in one launch, restarting at ``cu_seqlens`` boundaries (then ``B == 1``): what the layer's
    ``ShortConvolution`` modules compute on a fresh sequence (nha_fla/layers/nha.py:186-206).  Differentiable with
    respect to x, weight and bias."""
    _need_cuda(x, weight, bias)
    if activation not in (None, "silu", "swish"):
        raise ValueError(f"activation must be None, 'silu' or 'swish', got {activation!r}")
    if x.dim() != 3:
        raise ValueError(f"x must be [batch, tokens, channels], got {tuple(x.shape)}")
    Cn = x.shape[-1]
    if weight.shape[0] != Cn or weight.numel() != Cn * weight.shape[-1]:
        raise ValueError(f"weight must be [{Cn}, 1, taps] for x with {Cn} channels, got {tuple(weight.shape)}")
    if bias is not None and bias.numel() != Cn:
        raise ValueError(f"bias must have {Cn} entries, got {tuple(bias.shape)}")
    if cu_seqlens is not None and x.shape[0] != 1:
        raise ValueError("cu_seqlens needs the packed layout [1, T_tot, C]")
    if cu_seqlens is not None:
        # the kernels walk the boundaries: they must start at 0, not decrease and end at the token count
        cu_host = _cu_to_host(cu_seqlens)
        if cu_host.ndim != 1 or cu_host.size < 2 or cu_host[0] != 0 or cu_host[-1] != x.shape[1] \
                or (np.diff(cu_host) < 0).any():
            raise ValueError(f"cu_seqlens must rise from 0 to the token count {x.shape[1]}, got {cu_host.tolist()[:8]}"
                             f"{'...' if cu_host.size > 8 else ''}")
    cu = None if cu_seqlens is None else cu_seqlens.to(device=x.device, dtype=torch.int32).contiguous()
    return _ShortConvFunction.apply(x.contiguous(), weight, bias, cu, 0 if activation is None else 1)


def hybrid_prologue_supported(q: torch.Tensor, D: int, M: int) -> bool:
    """Whether nha_hybrid_prologue serves these tensors: GPU, bf16 / fp32, head size 64 / 128 / 256, M a multiple of 8."""
    return q.is_cuda and q.dtype in (torch.bfloat16, torch.float32) and D in (64, 128, 256) and M % 8 == 0


def _row_view(x: torch.Tensor, width: int, what: str):
    """(tensor, elements between the rows of two tokens) of a `[B, T, width]` view whose rows are contiguous and
    whose tokens are evenly spaced (a column slice of a fused projection output, or a contiguous tensor)."""
    B, T = x.shape[0], x.shape[1]
    if x.dim() != 3 or x.shape[2] != width:
        raise ValueError(f"{what} must be [batch, tokens, {width}], got {tuple(x.shape)}")
    if (width > 1 and x.stride(2) != 1) or (B > 1 and T > 1 and x.stride(0) != T * x.stride(1)):
        x = x.contiguous()
    stride = x.stride(1) if T > 1 else (x.stride(0) if B > 1 else width)
    esz = x.element_size()
    if (stride * esz) % 16 or x.data_ptr() % 16:
        x = x.contiguous()
        stride = width
    return x, stride


@torch.no_grad()
def nha_hybrid_prologue(q, k, v, f, cos, sin, *, num_heads: int, num_kv_heads: int, head_dim: int, num_slots: int,
                        q_weight=None, k_weight=None, eps: float = 1e-6, mask=None, gate_logit_normalizer: float = 8.0,
                        want_s: bool = True, positions=None, inv_freq=None):
    """One launch for the glue of a hybrid decoder attention block (inference): per-head RMSNorm of q and k (when
    weights are given), rotary embedding, the gates and the padding mask
    (nha_fla/models/qwen3_moe_nha/qwennha.py:103-144, :240-247).  q / k / v / f are `[B, T, heads * dim]` views
    (column slices of one fused projection output are read in place); cos / sin `[B or 1, T, D]`, or None with
    `positions [B, T]` (int64) and `inv_freq [D/2]` (fp32), from which the kernel forms the table rows itself; mask
    `[B, T]` or None; f None writes g = s = 0.  Returns contiguous q, sq `[B,T,HQ,D]`, k, sk, v `[B,T,H,D]`, g, s `[B,T,H,M]`
    (s None unless `want_s`)."""
    _need_cuda(q, k, v, cos, sin, positions, inv_freq)
    B, T = q.shape[0], q.shape[1]
    HQ, H, D, M = num_heads, num_kv_heads, head_dim, num_slots
    dt, dev = q.dtype, q.device
    if (cos is None) == (positions is None):
        raise ValueError("pass either cos and sin or positions and inv_freq")
    q, qs = _row_view(q, HQ * D, "q")
    k, ks = _row_view(k, H * D, "k")
    v, vs = _row_view(v, H * D, "v")
    fs = 0
    if f is not None:
        f, fs = _row_view(f, H * M, "f")
    cs_stride = 0
    if cos is not None:
        if cos.shape[-1] != D or cos.shape[-2] != T or cos.shape[0] not in (1, B) or sin.shape != cos.shape:
            raise ValueError(f"cos / sin must be [{B} or 1, {T}, {D}], got {tuple(cos.shape)} / {tuple(sin.shape)}")
        cos, sin = cos.to(dt).contiguous(), sin.to(dt).contiguous()
        cs_stride = T * D if cos.shape[0] == B and B > 1 else 0
    else:
        if tuple(positions.shape) != (B, T) or inv_freq.numel() != D // 2:
            raise ValueError(f"positions must be [{B}, {T}] and inv_freq [{D // 2}], got {tuple(positions.shape)} / "
                             f"{tuple(inv_freq.shape)}")
        positions = positions.to(torch.int64).contiguous()
        inv_freq = inv_freq.to(torch.float32).contiguous()
    for x in (k, v, f, q_weight, k_weight):
        if x is not None and x.dtype != dt:
            raise ValueError(f"every tensor must have the dtype of q ({dt}), got {x.dtype}")
    if mask is not None:
        mask = mask.reshape(B * T).to(dt).contiguous()
    new = lambda h, d: torch.empty(B, T, h, d, dtype=dt, device=dev)
    qo, sqo, ko, sko, vo, go = new(HQ, D), new(HQ, D), new(H, D), new(H, D), new(H, D), new(H, M)
    so = new(H, M) if want_s else None
    qw, kw = (None if w is None else w.contiguous() for w in (q_weight, k_weight))
    args = _lib.pack_hybrid_prologue(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), _at(f), qs, ks, vs, fs, _at(qw), _at(kw), _at(cos), _at(sin), cs_stride,
        _at(positions), _at(inv_freq), _at(mask), qo.data_ptr(), sqo.data_ptr(), ko.data_ptr(), sko.data_ptr(), vo.data_ptr(),
        go.data_ptr(), _at(so), B, T, HQ, H, D, M, _dtype_code(q), _lib.f32(float(eps)), _lib.f32(float(gate_logit_normalizer)),
        _stream(dev))
    _lib.check(_lib.load().hybrid_prologue_packed(args))
    return qo, sqo, ko, sko, vo, go, so


def zero_sink_attention_supported(q: torch.Tensor, k: torch.Tensor) -> bool:
    """Whether nha_sink_window_fwd serves these tensors: GPU, bf16, head size 64 or 128, a multiple of four query heads
    per kv-head, tensors of one call below 4 GiB."""
    HQ, H, D = q.shape[-2], k.shape[-2], q.shape[-1]
    tokens = q.numel() // (HQ * D)
    return (q.is_cuda and q.dtype == torch.bfloat16 and D in (64, 128) and HQ % H == 0 and (HQ // H) % 4 == 0
            and tokens * H * D * 2 < (1 << 32) and tokens <= 65535 * CHUNK)


@torch.no_grad()
def zero_sink_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, window: int, num_sinks: int,
                        scale: Optional[float] = None, cu_seqlens: Optional[torch.Tensor] = None,
                        output_lse: bool = False):
    """Sliding-window softmax attention preceded by `num_sinks` all-zero key / value rows per sequence: the "full
    attention" layers of the hybrid decoder models (nha_fla/models/qwen3_moe_nha/qwennha.py:323-336, :400-413).  q
    `[B,T,HQ,D]` and k, v `[B,T,H,D]` (rotated q / k; `[1,T_tot,...]` with cu_seqlens); query t of a sequence sees keys
    t - window < j <= t and clamp(window - 1 - t, 0, num_sinks) sinks of logit 0 and value 0.  One launch of the
    prefill's window loop.  Returns o `[B,T,HQ,D]` (and the log of the softmax denominator `[B,T,HQ]`)."""
    _need_cuda(q, k, v)
    if not zero_sink_attention_supported(q, k):
        raise _lib.NhaError(_lib.NHA_ERR_UNSUPPORTED, "zero_sink_attention: bf16, head size 64 / 128 and a multiple of four "
                                                       "query heads per kv-head are served")
    B, T, HQ, D = q.shape
    H = k.shape[2]
    if cu_seqlens is not None:
        if B != 1:
            raise ValueError("cu_seqlens needs the packed layout [1, T_tot, ...]")
        cu_host = _cu_to_host(cu_seqlens)
    else:
        cu_host = np.arange(0, (B + 1) * T, T, dtype=np.int32)
    if scale is None:
        scale = D ** -0.5
    dev = q.device
    q_, k_, v_ = (_flat(x) for x in (q, k, v))
    cu_d, idx_d, off_d, NT = prefill_tables(cu_host, dev)
    o = torch.empty(B * T, HQ, D, dtype=q.dtype, device=dev)
    lse = torch.empty(B * T, HQ, dtype=torch.float32, device=dev) if output_lse else None
    a = _lib.NhaSinkWindowArgs(q=_ptr(q_), k=_ptr(k_), v=_ptr(v_), o=_ptr(o), lse=_ptr(lse), cu_seqlens=_ptr(cu_d),
                               chunk_indices=_ptr(idx_d), chunk_offsets=_ptr(off_d), T_tot=B * T, N=cu_host.size - 1, NT=NT,
                               HQ=HQ, H=H, D=D, window=int(window), sinks=int(num_sinks), dtype=_dtype_code(q),
                               scale=float(scale), stream=_stream(dev))
    _lib.check(_lib.load().nha_sink_window_fwd(C.byref(a)))
    o = o.view(B, T, HQ, D)
    return (o, lse.view(B, T, HQ)) if output_lse else o


@torch.no_grad()
def nha_zero_sink_rescale_(o: torch.Tensor, lse_swa: torch.Tensor, window: int, num_sinks: int) -> torch.Tensor:
    """In place: row (b, t, head) of ``o [B,T,HQ,D]`` times (e^lse + num_sinks) / (e^lse + clamp(window - 1 - t, 0,
    num_sinks)) -- takes the zero-logit sinks that the NHA kernel's zero slot states put into every softmax back out
    where the reference's window no longer covers them (nha_fla/models/qwen3_moe_nha/qwennha.py:323-336)."""
    _need_cuda(o, lse_swa)
    B, T, HQ, D = o.shape
    if not o.is_contiguous() or lse_swa.dtype != torch.float32 or not lse_swa.is_contiguous() or tuple(lse_swa.shape) != (B, T, HQ):
        raise ValueError("o must be contiguous [B,T,HQ,D] and lse_swa contiguous fp32 [B,T,HQ]")
    lib = _lib.load()
    _lib.check(lib.nha_zero_sink_rescale(_ptr(o), _ptr(lse_swa), B, T, HQ, D, int(window), int(num_sinks), _dtype_code(o),
                                         _stream(o.device)))
    return o


class _ChunkNHAFunction(torch.autograd.Function):
    """Autograd node of chunk_nha on [B, T, heads, dim] tensors: same outputs (packed) and gradient set as
    ChunkNativeHybridAttentionFunction (nha_fla/ops/nha/chunk.py:364-564)."""

    @staticmethod
    def forward(ctx, q_swa, k_swa, q_gsa, k_gsa, v, s, g, h0k, h0v, cu_host, wl, shift, scale, want_state, impl):
        args = (q_swa, k_swa, q_gsa, k_gsa, v, s, g)
        args = [x.contiguous() for x in args]      # saved as they are: a view made here would hide later edits from autograd
        h0 = None if h0k is None else (h0k, h0v)
        o, lse_swa, lse_gsa, hkt, hvt = _prefill(args, (q_swa.shape[0] * q_swa.shape[1],), cu_host, wl, shift, scale, h0, want_state,
                                                 True, impl)
        ctx.save_for_backward(*args, o, lse_swa, lse_gsa, h0k, h0v)
        ctx.cu_host, ctx.wl, ctx.shift, ctx.scale = cu_host.copy(), wl, shift, scale    # it may be the caller's memory
        ctx.set_materialize_grads(False)
        if not want_state:
            return o, lse_swa, lse_gsa, None, None
        return o, lse_swa, lse_gsa, hkt, hvt

    @staticmethod
    @_first_derivatives_only
    def backward(ctx, do, dlse_swa, dlse_gsa, dhkt, dhvt):
        *args, o, lse_swa, lse_gsa, h0k, h0v = ctx.saved_tensors
        if do is None:
            do = torch.zeros_like(o)
        want_dh0 = h0k is not None and (ctx.needs_input_grad[7] or ctx.needs_input_grad[8])
        dht = None if dhkt is None and dhvt is None else (dhkt, dhvt)
        grads = _prefill_bwd([x.contiguous() for x in args], o, lse_swa, lse_gsa, do, ctx.cu_host, ctx.wl, ctx.shift, ctx.scale,
                             None if h0k is None else (h0k, h0v), dlse_swa, dlse_gsa, dht, want_dh0)
        dh0k, dh0v = grads[7], grads[8]
        if dh0k is not None:
            dh0k, dh0v = dh0k.to(h0k.dtype), dh0v.to(h0v.dtype)
        return (*grads[:7], dh0k, dh0v, None, None, None, None, None, None)


def _plain_autograd(tensors) -> bool:
    """Whether nothing but reverse-mode autograd looks at this call: ordinary tensors, no dispatch or function mode (fake
    tensors, operator counters), no functorch transform, no tracer, no forward-mode level."""
    return (all(t is None or type(t) in (torch.Tensor, torch.nn.Parameter) for t in tensors)
            and torch._C._len_torch_dispatch_stack() == 0 and not torch._C._is_torch_function_mode_enabled()
            and torch._C._functorch.peek_interpreter_stack() is None and torch._C._get_tracing_state() is None
            and torch.autograd.forward_ad._current_level < 0)


def _flat(x):
    return x.reshape(x.shape[0] * x.shape[1], *x.shape[2:]).contiguous()


@torch.compiler.disable
def chunk_nha(
    q_swa: torch.Tensor,
    k_swa: torch.Tensor,
    q_gsa: torch.Tensor,
    k_gsa: torch.Tensor,
    v: torch.Tensor,
    s: torch.Tensor,
    g: torch.Tensor,
    cu_seqlens: Optional[torch.Tensor] = None,
    max_seqlen: Optional[int] = None,
    scale: Optional[float] = None,
    window_size_left: int = -1,
    window_size_right: int = -1,
    head_first: Optional[bool] = False,
    gsa_kv_shift: int = 0,
    initial_state: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    output_final_state: bool = False,
    impl: Optional[str] = None,
):
    r"""Chunk-level Native Hybrid Attention forward (nha_fla/ops/nha/chunk.py:568-690).

    q_swa/q_gsa ``[B,T,HQ,D]``; k_swa/k_gsa ``[B,T,H,D]``, v ``[B,T,H,V]``, s/g ``[B,T,H,M]`` with
    ``HQ % H == 0`` (the reference takes ``H == HQ``).  ``cu_seqlens`` ``[N+1]`` selects varlen
    packing (then ``B == 1``).  The SWA branch is causal: ``window_size_right`` is accepted and
    has no effect, as in the reference's ``causal=True`` flash-attn call (chunk.py:423-431).
    Returns ``(o [B,T,HQ,V], lse_swa [B,T,HQ], lse_gsa [B,T,HQ])`` plus ``(hkt [N,H,K,M],
    hvt [N,H,M,V])`` fp32 when ``output_final_state`` (chunk.py:688-690).
    """
    if head_first:
        raise DeprecationWarning(
            "head_first is deprecated and will be removed in a future version. "
            "Please use head_first=False for now instead.",
        )
    assert q_swa.dim() == 4, "Expected [B, T, H, D] for input"
    _need_cuda(q_swa, k_swa, q_gsa, k_gsa, v, s, g)
    if q_swa.dtype == torch.float16:
        # float16 tensors: computed in float32 (every float16 value is one) by the kernels of that type, o returned in float16
        out = chunk_nha(*(x.float() for x in (q_swa, k_swa, q_gsa, k_gsa, v, s, g)), cu_seqlens=cu_seqlens, max_seqlen=max_seqlen,
                        scale=scale, window_size_left=window_size_left, window_size_right=window_size_right, head_first=head_first,
                        gsa_kv_shift=gsa_kv_shift, initial_state=initial_state, output_final_state=output_final_state, impl=impl)
        return (out[0].to(torch.float16), *out[1:])
    B, T, HQ, D = q_swa.shape
    H = k_swa.shape[2]
    if scale is None:
        scale = D ** -0.5
    if HQ % H:
        raise ValueError(f"query heads ({HQ}) must be a multiple of kv heads ({H})")
    for name, x, hh in (("q_gsa", q_gsa, HQ), ("k_gsa", k_gsa, H), ("v", v, H), ("s", s, H), ("g", g, H)):
        if x.shape[0] != B or x.shape[1] != T or x.shape[2] != hh:
            raise ValueError(f"{name} has shape {tuple(x.shape)}, expected [{B},{T},{hh},*]")
    if cu_seqlens is not None:
        if B != 1:
            raise ValueError("varlen (cu_seqlens) inputs must be packed with batch size 1")
        cu_host = _cu_to_host(cu_seqlens)
        if int(cu_host[-1]) != T:
            raise ValueError(f"cu_seqlens[-1] = {int(cu_host[-1])} does not match the packed length {T}")
    else:
        cu_host = np.arange(0, (B + 1) * T, T, dtype=np.int32)          # chunk.py:660
    dt = q_swa.dtype
    args = [x if x.dtype == dt else x.to(dt) for x in (q_swa, k_swa, q_gsa, k_gsa, v, s, g)]
    h0 = (None, None) if initial_state is None or initial_state[0] is None else tuple(initial_state)
    # empty sequences (a fully padded batch row after unpadding yields a repeated cu_seqlens entry): the
    # kernels see the packing without them; their final state is their initial state
    keep = None
    lens = None if cu_seqlens is None else np.diff(cu_host)
    if lens is not None and (lens < 0).any():
        raise ValueError("cu_seqlens must be non-decreasing")
    if lens is not None and (lens == 0).any():
        keep = torch.from_numpy(np.nonzero(lens > 0)[0]).to(q_swa.device)
        n_all = lens.size
        cu_host = np.concatenate([[0], np.cumsum(lens[lens > 0])]).astype(np.int32)
        h0_all = h0
        if h0[0] is not None:
            h0 = (h0[0][keep], h0[1][keep])
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (*args, *h0)):
        # the autograd node itself where nothing else has to see the call: the registered operator's dispatch costs a
        # training step 110 us of host time, where the GPU takes 210 to 270 for 1700 tokens
        if impl is not None or _plain_autograd((*args, *h0)):
            o, lse_swa, lse_gsa, hkt, hvt = _ChunkNHAFunction.apply(
                *args, h0[0], h0[1], cu_host, int(window_size_left), int(gsa_kv_shift), float(scale), output_final_state, impl)
        else:
            # the registered operator (nha_amd/custom_ops.py): schema, fake-tensor shapes and autograd formula
            o, lse_swa, lse_gsa, hkt, hvt = torch.ops.nha_amd.prefill_fwd(
                *(_flat(x) for x in args), torch.from_numpy(np.ascontiguousarray(cu_host, dtype=np.int32)), int(window_size_left),
                int(gsa_kv_shift), float(scale), h0[0], h0[1], bool(output_final_state))
    else:
        o, lse_swa, lse_gsa, hkt, hvt = _prefill([x.contiguous() for x in args], (B, T), cu_host, window_size_left, gsa_kv_shift, scale,
                                                 None if h0[0] is None else h0, output_final_state, True, impl)
    if keep is not None and output_final_state:
        def spread(part, init):
            full = torch.zeros(n_all, *part.shape[1:], dtype=part.dtype, device=part.device) if init is None \
                else init.to(part.dtype).clone()
            return full.index_copy(0, keep, part)
        hkt, hvt = spread(hkt, h0_all[0]), spread(hvt, h0_all[1])
    if o.dim() == 3:
        o, lse_swa, lse_gsa = o.view(B, T, HQ, -1), lse_swa.view(B, T, HQ), lse_gsa.view(B, T, HQ)
    if output_final_state:
        return o, lse_swa, lse_gsa, (hkt, hvt)
    return o, lse_swa, lse_gsa


@torch.no_grad()
def fused_chunk_nha_prefill(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    rotary_q: torch.Tensor,
    rotary_k: torch.Tensor,
    s: torch.Tensor,
    g: torch.Tensor,
    window_size: int,
    initial_state: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    output_final_state: bool = False,
    scale: Optional[float] = None,
    impl: Optional[str] = None,
) -> Tuple[torch.Tensor, Tuple[Optional[torch.Tensor], Optional[torch.Tensor]]]:
    r"""Fused NHA prefill, inference only (nha_fla/ops/nha/chunk_fused.py:291-380): window covers
    raw tokens ``[t-W+1, t]``, the slots hold tokens ``<= t-W``.  q/rotary_q ``[B,T,HQ,K]``;
    k/rotary_k/v/s/g ``[B,T,H,*]``.  Returns ``(o [B,T,HQ,V], (hkt, hvt))`` (Nones unless
    ``output_final_state``).  The reference's limits ``W <= 64`` and power-of-two dims <= 128
    (:331-332) do not apply here."""
    B, T, HQ, K = q.shape
    H = k.shape[2]
    W = int(window_size)
    assert k.shape[1] == T and v.shape[1] == T and s.shape[1] == T and g.shape[1] == T
    assert rotary_q.shape == q.shape and rotary_k.shape == k.shape
    assert HQ % H == 0
    assert W >= 1
    _need_cuda(q, k, v, rotary_q, rotary_k, s, g)
    if q.dtype == torch.float16:   # computed in float32, o returned in float16
        o, st = fused_chunk_nha_prefill(*(x.float() for x in (q, k, v, rotary_q, rotary_k, s, g)), window_size=window_size,
                                        initial_state=initial_state, output_final_state=output_final_state, scale=scale, impl=impl)
        return o.to(torch.float16), st
    if initial_state is not None and initial_state[0] is not None:
        hk0, hv0 = initial_state
        assert tuple(hk0.shape) == (B, H, K, s.shape[-1]) and tuple(hv0.shape) == (B, H, s.shape[-1], v.shape[-1]), \
            f"initial_state must be at the kv-head count [B, {H}, ...], got {tuple(hk0.shape)} / {tuple(hv0.shape)}"
    else:
        initial_state = None
    if scale is None:
        scale = K ** -0.5
    cu_host = np.arange(0, (B + 1) * T, T, dtype=np.int32)
    dt = q.dtype
    args = [_as(x, dt) for x in (rotary_q, rotary_k, q, k, v, s, g)]
    o, _, _, hkt, hvt = _prefill(args, (B, T), cu_host, W - 1, W, scale, initial_state, output_final_state, False, impl)
    return o, (hkt, hvt)


def _decode_state(initial_state, output_final_state, NG, B, H, K, V, M, dev):
    """State plumbing shared by the two T == 1 ops (fused_recurrent.py:169-179, :533-545)."""
    if initial_state is not None and initial_state[0] is not None:
        hk0, hv0 = initial_state
        if hk0.dtype != torch.float32 or hv0.dtype != torch.float32:
            raise TypeError("the slot state must be float32")
        hk0, hv0 = hk0.contiguous(), hv0.contiguous()
        assert tuple(hk0.shape) == (B, H, K, M) and tuple(hv0.shape) == (B, H, M, V), \
            f"initial_state must be ([{B},{H},{K},{M}], [{B},{H},{M},{V}]), got {tuple(hk0.shape)} / {tuple(hv0.shape)}"
    else:
        hk0 = hv0 = None
    hkt = hvt = None
    if output_final_state:
        if NG == 1 and hk0 is not None:
            hkt, hvt = hk0, hv0                                          # in place, as the reference
        else:
            hkt = torch.empty(B, H, K, M, dtype=torch.float32, device=dev)
            hvt = torch.empty(B, H, M, V, dtype=torch.float32, device=dev)
    return hk0, hv0, hkt, hvt


def fused_recurrent_nha_decode(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    g: torch.Tensor,
    sw_k: torch.Tensor,
    sw_v: torch.Tensor,
    sq: Optional[torch.Tensor] = None,
    s: Optional[torch.Tensor] = None,
    cos: Optional[torch.Tensor] = None,
    sin: Optional[torch.Tensor] = None,
    initial_state: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    output_final_state: bool = False,
    scale: Optional[float] = None,
) -> Tuple[torch.Tensor, Tuple[Optional[torch.Tensor], Optional[torch.Tensor]]]:
    r"""Single-token fused NHA decode step with GQA (nha_fla/ops/nha/fused_recurrent.py:431-584).

    q ``[B,1,HQ,K]`` raw; popped k/v/g ``[B,1,H,*]``; ``sw_k/sw_v [B,W,H,*]`` ascending in time;
    either ``sq`` (pre-rotated, with pre-rotated ``sw_k``) or ``cos/sin [B|1, W2>=W, K]``
    (in-kernel rotate-half on raw ``q``/``sw_k``; last W rows used, row W-1 = query position).
    Returns ``(o [B,1,HQ,V], (hkt, hvt))``; the state is updated in place when ``HQ == H``."""
    B, T, HQ, K = q.shape
    H = sw_k.shape[2]
    V = v.shape[-1]
    M = g.shape[-1]
    W = sw_k.shape[1]
    assert T == 1 and k.shape[1] == 1 and g.shape[1] == 1
    assert k.shape[2] == H and v.shape[2] == H and g.shape[2] == H, \
        f"popped-entry head count must match the kv-head count ({H}) of the window tensors"
    assert sw_v.shape[1] == W and sw_v.shape[2] == H
    assert HQ % H == 0
    assert K >= 16 and V >= 16
    _need_cuda(q, k, v, g, sw_k, sw_v, sq, s, cos, sin)
    if q.dtype == torch.float16:   # computed in float32, o returned in float16
        f = lambda x: None if x is None else x.float()
        o, st = fused_recurrent_nha_decode(f(q), f(k), f(v), f(g), f(sw_k), f(sw_v), sq=f(sq), s=f(s), cos=f(cos), sin=f(sin),
                                           initial_state=initial_state, output_final_state=output_final_state, scale=scale)
        return o.to(torch.float16), st
    NG = HQ // H
    if scale is None:
        scale = K ** -0.5
    dt = q.dtype
    rotary = cos is not None
    c_sb = c_sw = 0
    if rotary:
        assert sq is None, "pass either sq (pre-rotated) or cos/sin (in-kernel rotary), not both"
        assert sin is not None and cos.shape == sin.shape
        assert cos.shape[0] in (1, B) and cos.shape[1] >= W and cos.shape[2] == K, \
            f"rotary cos/sin must be [1|{B}, W2>={W}, K={K}], got {tuple(cos.shape)}"
        assert K % 2 == 0, "in-kernel rotate-half requires an even head dim"
        if cos.shape[1] > W:
            cos, sin = cos[:, -W:], sin[:, -W:]
        cos, sin = _as(cos, dt), _as(sin, dt)
        c_sb = cos.stride(0) if cos.shape[0] == B else 0
        c_sw = cos.stride(1)
    else:
        assert sq is not None and sq.shape == q.shape
    if s is not None:
        assert s.shape == g.shape
    dev = q.device
    q_, sq_, k_, v_, g_, s_, swk_, swv_ = (_as(x, dt) for x in (q, sq, k, v, g, s, sw_k, sw_v))
    hk0, hv0, hkt, hvt = _decode_state(initial_state, output_final_state, NG, B, H, K, V, M, dev)
    o = torch.empty(B, 1, HQ, V, dtype=dt, device=dev)
    stream = _stream(dev)
    scratch = decode_scratch(dev, stream)
    p = lambda x: 0 if x is None else x.data_ptr()
    args = _lib.pack_decode(
        _lib.NHA_DECODE_WINDOW, _dtype_code(q_), B, HQ, H, K, V, M, W, float(scale), p(q_), p(sq_), p(k_), p(v_), p(g_), p(s_),
        p(swk_), p(swv_), p(cos), p(sin), c_sb, c_sw, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, p(hk0), p(hv0), p(hkt), p(hvt), p(o),
        stream, 0, p(scratch), 0 if scratch is None else scratch.numel())
    run_decode(args, dev, scratch)
    return o, (hkt, hvt)


@torch.compiler.disable
def fused_recurrent_nha(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    sliding_window: torch.Tensor,
    s: torch.Tensor,
    g: torch.Tensor,
    scale: Optional[float] = None,
    initial_state: Optional[Tuple[torch.Tensor]] = None,
    output_final_state: Optional[bool] = False,
) -> Tuple[torch.Tensor, torch.Tensor, list]:
    r"""Single-token NHA inference step with caller-supplied window logits
    (nha_fla/ops/nha/fused_recurrent.py:588-682).  q ``[B,1,HQ,K]``; k/v/s/g ``[B,1,H,*]``;
    ``sliding_window [B,1,HQ,W]`` logits.  Returns ``(o [B,1,HQ,V]`` slot part only,
    ``swa_score [B,1,HQ,W]`` fp32 window probabilities of the mixing softmax, ``[hkt, hvt])``."""
    T = q.shape[1]
    if T != 1:
        raise ValueError(
            f"fused_recurrent_nha is the single-token inference path and expects T == 1, got T = {T}."
        )
    assert not q.requires_grad, "fused_recurrent_nha is inference-only (no autograd)"
    _need_cuda(q, k, v, sliding_window, s, g)
    if q.dtype == torch.float16:   # computed in float32, o returned in float16
        o, p, st = fused_recurrent_nha(q.float(), k.float(), v.float(), sliding_window.float(), s.float(), g.float(), scale=scale,
                                       initial_state=initial_state, output_final_state=output_final_state)
        return o.to(torch.float16), p, st
    if scale is None:
        scale = k.shape[-1] ** -0.5
    B, _, HQ, K = q.shape
    H, V, M, W = k.shape[2], v.shape[-1], s.shape[-1], sliding_window.shape[-1]
    assert HQ % H == 0
    NG = HQ // H
    dt = q.dtype
    dev = q.device
    cont = lambda x: x.to(dt).contiguous()
    q_, k_, v_, sw_, s_, g_ = map(cont, (q, k, v, sliding_window, s, g))
    hk0, hv0, hkt, hvt = _decode_state(initial_state, output_final_state, NG, B, H, K, V, M, dev)
    o = torch.empty(B, 1, HQ, V, dtype=dt, device=dev)
    probs = torch.empty(B, 1, HQ, W, dtype=torch.float32, device=dev)
    a = _lib.NhaDecodeArgs()
    a.mode, a.dtype = _lib.NHA_DECODE_LOGITS, _dtype_code(q_)
    a.B, a.HQ, a.H, a.K, a.V, a.M, a.W = B, HQ, H, K, V, M, W
    a.scale = float(scale)
    a.q = _ptr(q_)
    a.k_pop, a.v_pop, a.g_pop, a.s_pop = _ptr(k_), _ptr(v_), _ptr(g_), _ptr(s_)
    a.win_logits, a.win_probs = _ptr(sw_), _ptr(probs)
    a.hk_in, a.hv_in, a.hk_out, a.hv_out = _ptr(hk0), _ptr(hv0), _ptr(hkt), _ptr(hvt)
    a.o, a.stream = _ptr(o), _stream(dev)
    _lib.check(_lib.load().nha_decode_step(C.byref(a)))
    return o, probs, [hkt, hvt]
