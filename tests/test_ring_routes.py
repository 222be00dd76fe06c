"""Handing a prompt to a decode ring outside ordinary calls: the one-launch form steps aside for fake tensors, dispatch modes
and forward-mode differentiation, where the tensor operations answer."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


def _inputs(B=2, T=20, H=2, K=64, M=64, dtype=torch.bfloat16):
    r = lambda *s: torch.randn(*s, device="cuda").to(dtype)
    return [r(B, T, H, K), r(B, T, H, K), r(B, T, H, K), r(B, T, H, M)], (r(B, H, K, M).float(), r(B, H, M, K).float())


@pytest.mark.parametrize("packed", [False, True])
def test_fake_tensors(packed):
    from nha_amd import NHARingState
    with FakeTensorMode():
        rows, state = _inputs(B=1 if packed else 2)
        st = NHARingState.from_prefill(*rows, state, 8, cu_seqlens=torch.empty(2, dtype=torch.int32, device="cuda") if packed else None)
    N = 1 if packed else 2
    assert st.ring_k.shape == (N, 8, 2, 64) and st.hk.shape == (N, 2, 64, 64) and st.count.shape == (N,) and st.count.dtype == torch.int32


@pytest.mark.gpu
def test_forward_mode_and_dispatch_modes():
    import torch.autograd.forward_ad as fwAD
    from torch.utils._python_dispatch import TorchDispatchMode
    from nha_amd import NHARingState
    rows, state = _inputs()
    want = NHARingState.from_prefill(*rows, state, 8)
    tangents = [torch.randn_like(x) for x in rows]
    with fwAD.dual_level():
        st = NHARingState.from_prefill(*[fwAD.make_dual(x, t) for x, t in zip(rows, tangents)], state, 8)
        rings = [fwAD.unpack_dual(x) for x in (st.ring_k, st.ring_kg, st.ring_v, st.ring_g)]
    moved = NHARingState.from_prefill(*tangents, state, 8)
    for ring, t, w in zip(rings, (moved.ring_k, moved.ring_kg, moved.ring_v, moved.ring_g), (want.ring_k, want.ring_kg, want.ring_v, want.ring_g)):
        assert torch.equal(ring.primal, w) and torch.equal(ring.tangent, t)

    class Seen(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))
    with Seen() as mode:
        st = NHARingState.from_prefill(*rows, state, 8)
    assert any("gather" in n or "index" in n for n in mode.names) and torch.equal(st.ring_k, want.ring_k)
