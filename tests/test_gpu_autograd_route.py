"""chunk_nha reaches its autograd node directly for ordinary calls and through the registered operator where a dispatch
mode, a transform or a tensor subclass has to see it: both give the same outputs and gradients, bit for bit."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu
KEYS = ["q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g"]


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def _call(d, dtype=torch.bfloat16, cu=None, strided=False, state=False, hooks=False):
    from nha_amd import chunk_nha
    leaves = [d[k].cuda().to(torch.float32 if k == "g" and dtype is None else d[k].dtype) for k in KEYS]
    if strided:
        leaves = [torch.stack([x, x], -1)[..., 0] for x in leaves]
    leaves = [x.detach().requires_grad_() for x in leaves]
    h0 = tuple(t.cuda().requires_grad_() for t in d["h0"])
    seen = []
    hook = torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(1), t.cpu())[1], lambda t: t.cuda()) if hooks \
        else torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t)
    with hook:
        out = chunk_nha(*leaves, window_size_left=40, gsa_kv_shift=16, initial_state=h0, output_final_state=state,
                        cu_seqlens=None if cu is None else torch.tensor(cu, dtype=torch.int32).cuda())
    flat = [*out[:3], *(out[3] if state else ())]
    gen = torch.Generator().manual_seed(5)
    cot = [torch.randn(t.shape, generator=gen).to(t.dtype).cuda() for t in flat]
    grads = torch.autograd.grad(flat, [*leaves, *h0], cot)
    return flat, grads, seen


@pytest.mark.parametrize("kind", ["plain", "strided", "mixed types", "packed", "empty sequence"])
def test_both_routes_agree(kind):
    cu = {"packed": [0, 1, 66, 150], "empty sequence": [0, 70, 70, 150]}.get(kind)
    n = 2 if cu is None else 3
    d = prefill_inputs(77, 2 if cu is None else 1, 150, 4, 2, 64, 64, 64, qk_scale=0.125, with_state=True, N=n)
    kw = dict(cu=cu, strided=kind == "strided", state=True, dtype=None if kind == "mixed types" else torch.bfloat16)
    a_out, a_grad, _ = _call(d, **kw)
    with _Seen() as mode:
        b_out, b_grad, _ = _call(d, **kw)
    assert any("prefill_fwd" in x for x in mode.names) and any("prefill_bwd" in x for x in mode.names)
    for x, y in zip([*a_out, *a_grad], [*b_out, *b_grad]):
        assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)


def test_hooks_edits_and_second_derivatives():
    """Saved tensors pass the caller's hooks, an input edited in place after the call is noticed, and a second derivative
    is refused, not taken for zero."""
    from nha_amd import chunk_nha
    d = prefill_inputs(78, 1, 90, 4, 2, 64, 64, 64, qk_scale=0.125, with_state=True)
    _, plain, _ = _call(d)
    _, hooked, seen = _call(d, hooks=True)
    assert len(seen) >= 10 and all(torch.equal(x, y) for x, y in zip(plain, hooked))
    leaves = [d[k].cuda().requires_grad_() for k in KEYS]
    x = leaves[4] * 1
    o = chunk_nha(*leaves[:4], x, *leaves[5:], window_size_left=40)[0]
    with torch.no_grad():
        x.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.float().sum().backward()
    o = chunk_nha(*leaves, window_size_left=40)[0]
    gr = torch.autograd.grad(o.float().sum(), leaves[4], create_graph=True)[0]
    with pytest.raises(RuntimeError):
        gr.float().sum().backward()
