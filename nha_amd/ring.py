"""Resident decode state: fp32 slot state + W-slot K/V/gate ring buffers, stepped by ONE kernel.

Replaces the cat-shift window cache and the pop/update choreography around the decode op in the
reference (nha_fla/models/nha_cache.py:105-131, :143-154; models/qwen3_moe_nha/qwennha.py:151-176,
:351-365): the kernel pops the oldest ring entry into the slots, stores the new token in its
slot and attends over the valid entries, reading state and window once per kv-head."""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import torch

from . import _lib
from .ops import _dtype_code, _need_cuda, _plain_autograd, _ptr, _stream, decode_scratch, run_decode


@dataclass
class NHARingState:
    """Per-layer decode state for B sequences.  ``ring_k`` holds the window keys as the window
    branch reads them (already rotated), ``ring_kg`` the slot-branch keys (raw), ``ring_g`` the
    log forget gates of the cached tokens; ``count[b]`` tokens have been cached so far."""
    hk: torch.Tensor        # [B,H,K,M] fp32
    hv: torch.Tensor        # [B,H,M,V] fp32
    ring_k: torch.Tensor    # [B,W,H,K]
    ring_kg: torch.Tensor   # [B,W,H,K]
    ring_v: torch.Tensor    # [B,W,H,V]
    ring_g: torch.Tensor    # [B,W,H,M]
    count: torch.Tensor     # [B] int32; the tensor bound to this name changes with every step
    count_alt: Optional[torch.Tensor] = None   # the other counter array (the step writes count + 1 there)
    # the slots never absorb anything (every cached log-gate is 0 and every write strength 0: the zero-sink layers of
    # the hybrid models): hk and hv stay zero, and the step neither reads nor writes them
    zero_state: bool = False
    # the step's scratch, where it must not be the stream's shared one: a recorded step keeps its own (zeroed before the
    # recording, so that a replay need not clear it)
    scratch: Optional[torch.Tensor] = None

    @classmethod
    def empty(cls, B, H, K, V, M, W, dtype=torch.bfloat16, device="cuda") -> "NHARingState":
        z = lambda *s, dt=dtype: torch.zeros(*s, dtype=dt, device=device)
        return cls(z(B, H, K, M, dt=torch.float32), z(B, H, M, V, dt=torch.float32), z(B, W, H, K), z(B, W, H, K),
                   z(B, W, H, V), z(B, W, H, M), z(B, dt=torch.int32))

    @classmethod
    def from_prefill(cls, k_swa, k_gsa, v, g, final_state, window: int, cu_seqlens=None) -> "NHARingState":
        """The decode state that continues a prefill with ``(window_size_left, gsa_kv_shift) =
        (window - 1, window)``: the slot state is the prefill's final state (it has absorbed the
        tokens that left the window), ring slot ``j % window`` holds token ``j`` for the last
        ``min(L, window)`` tokens of each sequence and ``count = L``.  Takes the prefill's own
        operands: k_swa (rotated), k_gsa, v ``[B,T,H,*]``, g ``[B,T,H,M]`` (``[1,T_tot,...]`` with
        cu_seqlens) and ``final_state = (hk [N,H,K,M], hv [N,H,M,V])``.  The hand-over the reference
        does by slicing the last ``window`` rows into its cache (nha_fla/models/nha_cache.py:87-91)."""
        _need_cuda(k_swa, k_gsa, v, g, final_state[0], final_state[1])
        dev, W = k_swa.device, int(window)
        B, T, H, K = k_swa.shape
        V, M = v.shape[-1], g.shape[-1]
        hk, hv = final_state
        if cu_seqlens is not None and B != 1:
            raise ValueError("cu_seqlens needs the packed layout [1, T_tot, ...]")
        N = B if cu_seqlens is None else cu_seqlens.numel() - 1
        if tuple(hk.shape) != (N, H, K, M) or tuple(hv.shape) != (N, H, M, V):
            raise ValueError(f"final_state must be ([{N},{H},{K},{M}], [{N},{H},{M},{V}]), got {tuple(hk.shape)}, {tuple(hv.shape)}")
        st = cls._fill((k_swa, k_gsa, v, g), hk, hv, W, cu_seqlens, N, T)
        if st is not None:
            return st
        if cu_seqlens is None:
            starts = torch.arange(B, device=dev, dtype=torch.long) * T
            lens = torch.full((B,), T, device=dev, dtype=torch.long)
        else:
            cu = cu_seqlens.to(device=dev, dtype=torch.long)
            starts, lens = cu[:-1], cu[1:] - cu[:-1]
        r = torch.arange(W, device=dev, dtype=torch.long)
        last = (lens - 1)[:, None]
        tok = last - torch.remainder(last - r[None, :], W)            # newest token j <= L-1 with j % W == r
        valid = tok >= 0
        src = (starts[:, None] + tok.clamp_min(0)).reshape(-1)

        def gather(x):
            rows = x.reshape(B * T, *x.shape[2:]).index_select(0, src).reshape(N, W, *x.shape[2:])
            return rows * valid[:, :, None, None].to(rows.dtype)

        return cls(hk.to(torch.float32).clone(), hv.to(torch.float32).clone(), gather(k_swa), gather(k_gsa), gather(v),
                   gather(g), lens.to(torch.int32))

    @classmethod
    def _fill(cls, rows, hk, hv, W: int, cu_seqlens, N: int, T: int) -> Optional["NHARingState"]:
        """The hand-over in one launch, or None for what the kernel does not move: rows, states or addresses that are
        not whole 16-byte pieces, states that are not fp32, tensors with a gradient to carry or on several devices, calls that
        something besides autograd looks at (fake tensors, modes, forward-mode levels)."""
        dev = rows[0].device
        ts = (*rows, hk, hv)
        if (torch.compiler.is_compiling() or not _plain_autograd((*ts, cu_seqlens)) or N < 1 or N > 65535 or W < 1
                or any(x.dim() != 4 or x.shape[:2] != rows[0].shape[:2] or x.numel() == 0 for x in rows)
                or any(x.device != dev for x in ts) or dev.index != torch.cuda.current_device() or (torch.is_grad_enabled() and any(x.requires_grad for x in ts))
                or hk.dtype != torch.float32 or hv.dtype != torch.float32):
            return None
        rows, states = [x.contiguous() for x in rows], [hk.contiguous(), hv.contiguous()]
        rings = [x.new_empty(N, W, *x.shape[2:]) for x in rows]
        out = [torch.empty_like(x) for x in states]
        count = torch.empty(N, dtype=torch.int32, device=dev)
        cu = None if cu_seqlens is None else cu_seqlens.to(device=dev, dtype=torch.int32).contiguous()
        sizes = [x.shape[2] * x.shape[3] * x.element_size() for x in rows]
        state_sizes = [x.numel() // N * 4 for x in states]
        if any(b % 16 for b in (*sizes, *state_sizes)) or any(x.data_ptr() % 16 for x in (*rows, *states)):
            return None
        at = lambda xs: [x.data_ptr() for x in xs]
        args = _lib.pack_ring_fill(*at(rows), *at(rings), *sizes, *at(states), *at(out), *state_sizes, 0 if cu is None else cu.data_ptr(),
                                   count.data_ptr(), rows[0].shape[0] * T, N, T, _lib.i32(W), _stream(dev))
        _lib.check(_lib.load().ring_fill_packed(args))
        return cls(*out, *rings, count)

    @property
    def window(self) -> int:
        return self.ring_k.shape[1]


def ring_advance(state: NHARingState) -> None:
    """count += 1 for every sequence, in place (one small launch).  For steps taken with ``advance=False``: a
    captured HIP graph replays fixed pointers, so it cannot trade the two counter arrays as the eager step does;
    it runs the step on ``count`` and then this launch."""
    _lib.check(_lib.load().nha_decode_advance(_ptr(state.count), state.count.numel(), _stream(state.count.device)))


def ring_decode_step(state: NHARingState, q: torch.Tensor, sq: torch.Tensor, k_new: torch.Tensor,
                     kg_new: torch.Tensor, v_new: torch.Tensor, g_new: torch.Tensor,
                     scale: Optional[float] = None, out: Optional[torch.Tensor] = None,
                     advance: bool = True) -> torch.Tensor:
    """One decode step for every sequence of ``state`` (updated in place).

    q (slot-branch query) and sq (window query, rotated) ``[B,HQ,K]``; the new token's window key
    ``k_new`` (rotated), slot key ``kg_new`` ``[B,H,K]``, value ``[B,H,V]`` and log gate
    ``g_new [B,H,M]``.  Returns ``o [B,HQ,V]``."""
    _need_cuda(q, sq, k_new, kg_new, v_new, g_new, state.hk)
    B, HQ, K = q.shape
    _, W, H, _ = state.ring_k.shape
    V, M = state.ring_v.shape[-1], state.ring_g.shape[-1]
    dt = state.ring_k.dtype
    qshape, kshape = (B, HQ, K), (B, H, K)
    for name, x, shp in (("q", q, qshape), ("sq", sq, qshape), ("k_new", k_new, kshape), ("kg_new", kg_new, kshape),
                         ("v_new", v_new, (B, H, V)), ("g_new", g_new, (B, H, M))):
        if x.shape != shp or x.dtype != dt or not x.is_contiguous():
            raise ValueError(f"{name} must be a contiguous {dt} tensor of shape {shp}, got {tuple(x.shape)} {x.dtype}")
    if scale is None:
        scale = K ** -0.5
    dev = q.device
    o = out if out is not None else torch.empty(B, HQ, V, dtype=dt, device=dev)
    if advance and state.count_alt is None:
        state.count_alt = torch.empty_like(state.count)
    stream = _stream(dev)
    scratch = state.scratch if state.scratch is not None else decode_scratch(dev, stream)
    # NULL states (zero_state): the kernel takes zeros and writes nothing back
    hk, hv = (0, 0) if state.zero_state else (state.hk.data_ptr(), state.hv.data_ptr())
    args = _lib.pack_decode(
        _lib.NHA_DECODE_RING, _dtype_code(q), B, HQ, H, K, V, M, W, float(scale), q.data_ptr(), sq.data_ptr(), 0, 0, 0, 0, 0, 0,
        0, 0, 0, 0, 0, 0, state.ring_k.data_ptr(), state.ring_kg.data_ptr(), state.ring_v.data_ptr(), state.ring_g.data_ptr(),
        k_new.data_ptr(), kg_new.data_ptr(), v_new.data_ptr(), g_new.data_ptr(), state.count.data_ptr(), hk, hv, hk, hv,
        o.data_ptr(), stream, state.count_alt.data_ptr() if advance else 0,      # the kernel writes count + 1 there
        *((0, 0) if scratch is None else (scratch.data_ptr(), scratch.numel())))
    run_decode(args, dev, scratch)
    if advance:      # the two counter arrays trade places
        state.count, state.count_alt = state.count_alt, state.count
    return o
