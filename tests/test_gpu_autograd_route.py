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


NODES = ["operator", "prologue", "projections and prologue", "epilogue", "short convolution", "layer", "layer, short convolution"]


def _node(node):
    """A function of one tensor [1, 90, 128] to the scalar of one node's outputs."""
    from nha_amd import chunk_nha, ops
    from nha_amd.layer import NativeHybridAttention
    torch.manual_seed(2)
    r = lambda *s: torch.randn(*s, device="cuda").bfloat16()
    inv = 10000.0 ** (-torch.arange(0, 64, 2, device="cuda").float() / 64)
    total = lambda ts: sum(t.float().pow(2).sum() for t in ts)
    kw = dict(feature_map="swish", gate_logit_normalizer=8)
    heads = lambda x: [y.view(1, 90, 2, 64) for y in (x, x * 2, x * 3, x * 4)]
    if node.startswith("layer"):
        m = NativeHybridAttention(hidden_size=128, num_heads=2, num_slots=64, layer_idx=0, window_size=40, use_short_conv="short" in node)
        m = m.cuda().bfloat16()
        return lambda x: total(m(x)[:1])
    if node == "operator":
        s, g = r(1, 90, 2, 64).sigmoid(), -r(1, 90, 2, 64).abs()
        return lambda x: total((lambda q, k, v, f: chunk_nha(q, k, q, k, v, s, g, window_size_left=40)[:1])(*heads(x)))
    if node == "prologue":
        return lambda x: total(ops.nha_layer_prologue(*heads(x), inv, **kw))
    if node == "projections and prologue":
        mods = [torch.nn.Linear(128, 128, bias=False).cuda().bfloat16() for _ in range(4)]
        return lambda x: total(ops.nha_layer_prologue(None, None, None, None, inv, projections=(x, mods, (2, 2, 64, 64, 64)), **kw))
    w, taps = r(128).requires_grad_(), r(128, 4).requires_grad_()
    if node == "epilogue":
        return lambda x: total([ops.nha_layer_epilogue(x, w, None, 1e-5)])
    return lambda x: total([ops.nha_short_conv(x, taps, None, activation="silu")])


def _same(node, a, b):
    # the layer's projections add four products in another order where a graph is wanted: a rounding of 2^-8 each
    return torch.equal(a, b) if node != "layer, short convolution" else (a - b).float().norm() <= 1e-2 * b.float().norm()


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("node", NODES)
def test_second_derivatives_through_the_kernels_are_refused(node, residual):
    """The kernels have first derivatives only: a gradient taken with create_graph leads to an error, never to a second
    derivative without the terms that pass through them, whether the input is reached through them alone or past them too."""
    f = _node(node)
    x = torch.randn(1, 90, 128, device="cuda").bfloat16().requires_grad_()
    out = f(x)
    if residual:
        out = out + x.float().pow(3).sum()
    plain = torch.autograd.grad(out, x, retain_graph=True)[0]
    dx = torch.autograd.grad(out, x, create_graph=True)[0]
    assert dx.requires_grad and _same(node, dx, plain)
    with pytest.raises(RuntimeError, match="differentiated twice"):
        torch.autograd.grad(dx.float().pow(2).sum(), x)


@pytest.mark.parametrize("create_graph", [False, True])
@pytest.mark.parametrize("node", NODES)
def test_first_derivatives_under_checkpointing(node, create_graph):
    """Saved tensors that are formed anew in the backward are unpacked once, with and without a graph of the gradients."""
    from torch.utils.checkpoint import checkpoint
    f = _node(node)
    x = torch.randn(1, 90, 128, device="cuda").bfloat16().requires_grad_()
    plain = torch.autograd.grad(f(x), x)[0]
    dx = torch.autograd.grad(checkpoint(f, x, use_reentrant=False), x, create_graph=create_graph)[0]
    assert _same(node, dx, plain)
