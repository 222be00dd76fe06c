"""nha_wgrad (weight gradients of projections of one input) against the fp64 product, and the layer's shared projections
against its modules called one by one.  fp32 sums and one rounding to bf16 (8 significant bits), which is 2^-8 of the value at
most: relative L2 4e-3."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


# one token; one past a step of 64; columns of one 16-byte piece, around a tile of 256; splits that do not divide the tokens
@pytest.mark.parametrize("T,width,outs", [(1, 8, [8]), (65, 256, [256, 8]), (777, 520, [264, 248, 8]), (129, 248, [512]),
                                          (4099, 264, [256, 256, 64, 8]), (20000, 128, [136])])
def test_wgrad(T, width, outs):
    from nha_amd.ops import nha_wgrad
    gen = torch.Generator(device="cuda").manual_seed(T + width)
    x = torch.randn(T, width, generator=gen, device="cuda").bfloat16()
    dys = [torch.randn(T, o, generator=gen, device="cuda").bfloat16() for o in outs]
    for dy, dw in zip(dys, nha_wgrad(x, dys)):
        ref = dy.double().t() @ x.double()
        rel = ((dw.double() - ref).norm() / ref.norm()).item()
        assert rel <= 4e-3, f"{tuple(dw.shape)}: relative L2 error {rel:.3e}"


# units of 32 tokens, of which four lie in LDS: one token to five units, a token less and more
@pytest.mark.parametrize("T", [31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 160, 161])
def test_wgrad_few_units(T):
    """Tokens past the last one add nothing, whatever the last one holds: an infinite gradient stays infinite, and reaches its row
    of the weights only."""
    from nha_amd.ops import nha_wgrad
    gen = torch.Generator(device="cuda").manual_seed(T)
    x, dy = (torch.randn(T, n, generator=gen, device="cuda").bfloat16() for n in (264, 272))
    x[-1] = x[-1].abs() + 1
    dy[-1, 7] = float("inf")
    dw, = nha_wgrad(x, [dy])
    assert (dw[7] == float("inf")).all()
    rest = [i for i in range(272) if i != 7]
    ref = (dy.double().t() @ x.double())[rest]
    assert ((dw[rest].double() - ref).norm() / ref.norm()).item() <= 4e-3


def test_wgrad_row_stride():
    from nha_amd.ops import nha_wgrad
    gen = torch.Generator(device="cuda").manual_seed(9)
    x, both = (torch.randn(333, n, generator=gen, device="cuda").bfloat16() for n in (72, 344))
    dense = nha_wgrad(x, [both[:, :264].contiguous(), both[:, 264:].contiguous()])
    assert all(torch.equal(a, b) for a, b in zip(dense, nha_wgrad(x, [both[:, :264], both[:, 264:]])))


@pytest.mark.parametrize("case", ["dense beside columns", "columns beside dense", "two matrices", "expanded", "every second column", "x of a matrix"])
def test_wgrad_rows_of_different_strides(case):
    """Gradients whose rows do not lie one common stride apart, 16-byte pieces within them, are the same as dense ones."""
    from nha_amd.ops import nha_wgrad
    r = lambda *s: torch.randn(*s, device="cuda").bfloat16()
    x, wide, other = r(130, 72), r(130, 344), r(130, 64)
    dys = {"dense beside columns": [r(130, 64), wide[:, :264]], "columns beside dense": [wide[:, 264:], r(130, 64)],
           "two matrices": [wide[:, :64], other[:, 8:16]], "expanded": [r(1, 64).expand(130, 64), wide[:, :8]],
           "every second column": [wide[:, ::2][:, :64]], "x of a matrix": [r(130, 64)]}[case]
    if case == "x of a matrix":
        x = r(130, 144)[:, ::2]
    dense = nha_wgrad(x.contiguous(), [dy.contiguous() for dy in dys])
    assert all(torch.equal(a, b) for a, b in zip(dense, nha_wgrad(x, dys)))


def test_wgrad_refuses_tensors_that_do_not_fit():
    from nha_amd.ops import nha_wgrad
    x, dy = torch.randn(64, 32, device="cuda").bfloat16(), torch.randn(60, 16, device="cuda").bfloat16()
    for bad in ([dy], [], [dy] * 5):
        with pytest.raises(ValueError):
            nha_wgrad(x, bad)
    with pytest.raises(TypeError):
        nha_wgrad(x, [x.float()])


def test_wgrad_scratch_is_its_own(monkeypatch):
    """The partial sums lie between two launches: not in the workspace that every call of a stream shares, which another thread
    may queue a call on in between."""
    from nha_amd import ops
    monkeypatch.setattr(ops, "_workspace", lambda *a: pytest.fail("shared workspace"))
    x, dy = (torch.randn(500, n, device="cuda").bfloat16() for n in (64, 32))
    assert ops.nha_wgrad(x, [dy])[0].shape == (32, 64)


def test_wgrad_refuses():
    from nha_amd import _lib
    lib = _lib.load()
    a = _lib.NhaWgradArgs(n=1, T=64, I=12)
    a.O[0] = 8
    assert lib.nha_wgrad_scratch_bytes(C.byref(a)) == 0
    a.I, a.n = 16, 5
    assert lib.nha_wgrad_scratch_bytes(C.byref(a)) == 0
    a.n = 1
    assert lib.nha_wgrad_scratch_bytes(C.byref(a)) > 0 and lib.nha_wgrad(C.byref(a)) != 0      # no tensors


def _layer(**kw):
    from nha_amd.layer import NativeHybridAttention
    torch.manual_seed(4)
    return NativeHybridAttention(hidden_size=256, num_heads=4, num_kv_heads=2, num_slots=64, layer_idx=0, window_size=40,
                                 **kw).cuda().bfloat16()


@pytest.mark.parametrize("case", ["plain", "frozen", "short conv", "strided input", "padding mask", "frozen input"])
def test_layer_projections(case):
    layer = _layer(use_short_conv=case == "short conv")
    x = torch.randn(2, 90, 512 if case == "strided input" else 256, device="cuda").bfloat16()[..., :256].requires_grad_()
    if case == "frozen":
        layer.k_proj.weight.requires_grad_(False)
    if case == "frozen input":
        x = x.detach()
    kw = dict(attention_mask=(torch.arange(90)[None] >= torch.tensor([[0], [27]])).cuda()) if case == "padding mask" else {}
    leaves = [t for t in (x, *layer.parameters()) if t.requires_grad]
    dy = torch.randn(2, 90, 256, device="cuda").bfloat16()

    def run():
        y = layer(x, **kw)[0]
        return y, torch.autograd.grad(y, leaves, dy)
    y, grads = run()
    seen = []
    for m in (layer.q_proj, layer.f_proj):                 # a hook: the modules are called
        m.register_forward_hook(lambda *a: seen.append(1))
    y2, grads2 = run()
    # one product or four: the same sums in another order, one rounding of 2^-8 in q, k, v and f
    assert len(seen) == 2 and ((y.double() - y2.double()).norm() / y2.double().norm()).item() <= 1e-2
    for g, r in zip(grads, grads2):
        # dx adds four products in bf16 one way and inside the products the other: up to four roundings of 2^-8, independent of each other and of one quarter to all of the sum
        assert g.shape == r.shape and g.dtype == r.dtype
        assert ((g.double() - r.double()).norm() / r.double().norm()).item() <= 1e-2


def test_wide_layer_projections():
    """Weights past the size that nha_wgrad takes: the node's gradients are the library's."""
    from nha_amd.ops import nha_layer_prologue
    torch.manual_seed(8)
    modules = [torch.nn.Linear(4096, n, bias=False).cuda().bfloat16() for n in (4096, 1024, 1024, 512)]
    inv = 10000.0 ** (-torch.arange(0, 128, 2, device="cuda").float() / 128)
    x = torch.randn(2, 40, 4096, device="cuda").bfloat16().requires_grad_()
    leaves, grads = [x, *(m.weight for m in modules)], []
    kw = dict(feature_map="swish", gate_logit_normalizer=8)
    for one in (True, False):
        out = nha_layer_prologue(None, None, None, None, inv, projections=(x, modules, (32, 8, 128, 128, 64)), **kw) if one else \
            nha_layer_prologue(*(m(x).unflatten(-1, (h, -1)) for m, h in zip(modules, (32, 8, 8, 8))), inv, **kw)
        grads.append(torch.autograd.grad([t.float().pow(2).sum() for t in out], leaves))
    for a, b in zip(*grads):      # q, k, v, f from one product or four, dx of one or four: roundings of 2^-8
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() <= 1e-2


@pytest.mark.parametrize("case", ["no grad", "fp32"])
def test_calls_that_cannot_be_one_node_look_at_no_module(case, monkeypatch):
    from nha_amd import ops
    layer, seen = _layer().to(torch.float32 if case == "fp32" else torch.bfloat16), []
    monkeypatch.setattr(ops, "_plain_modules", lambda m: seen.append(m) or False)
    x = torch.randn(1, 50, 256, device="cuda", dtype=layer.q_proj.weight.dtype)
    with torch.set_grad_enabled(case != "no grad"):
        assert layer(x)[0].isfinite().all() and not seen


def test_second_derivative_of_the_projections():
    from nha_amd.ops import shared_input_linears
    lin = [torch.nn.Linear(64, o, bias=False).cuda().bfloat16() for o in (32, 16)]
    x = torch.randn(20, 64, device="cuda").bfloat16().requires_grad_()
    got, ref = [], []
    for out, call in ((got, lambda: shared_input_linears(x, lin)), (ref, lambda: [m(x) for m in lin])):
        a, b = call()
        dx = torch.autograd.grad((a.float().pow(2).sum() + b.float().pow(2).sum()), x, create_graph=True)[0]
        out.extend(torch.autograd.grad(dx.float().pow(2).sum(), [x, *(m.weight for m in lin)]))
    for g, r in zip(got, ref):
        assert ((g.double() - r.double()).norm() / r.double().norm()).item() <= 1e-2


def _front_call(modules, x, inv, fmap="swish", cu=None):
    from nha_amd.ops import nha_layer_prologue
    return nha_layer_prologue(None, None, None, None, inv, feature_map=fmap, gate_logit_normalizer=8, cu_seqlens=cu,
                              projections=(x, modules, (4, 2, 64, 64, 64)))


@pytest.mark.parametrize("case", ["one node", "no grad", "no feature map", "bias", "hook", "fp32"])
def test_prologue_on_projections(case):
    """The form that takes the projections gives what the plain form gives on the modules' outputs, also for calls that cannot
    be one node."""
    from nha_amd.ops import nha_layer_prologue
    torch.manual_seed(6)
    dt = torch.float32 if case == "fp32" else torch.bfloat16
    modules = [torch.nn.Linear(128, n, bias=case == "bias").cuda().to(dt) for n in (256, 128, 128, 128)]
    x = torch.randn(2, 50, 128, device="cuda").to(dt).requires_grad_()
    inv = 10000.0 ** (-torch.arange(0, 64, 2, device="cuda").float() / 64)
    fmap = None if case == "no feature map" else "swish"
    seen = []
    if case == "hook":
        modules[1].register_forward_hook(lambda *a: seen.append(1))
    with torch.set_grad_enabled(case != "no grad"):
        got = _front_call(modules, x, inv, fmap)
        raw = [m(x).unflatten(-1, (h, 64)) for m, h in zip(modules, (4, 2, 2, 2))]
        want = nha_layer_prologue(*raw, inv, feature_map=fmap, gate_logit_normalizer=8)
    for a, b in zip(got, want):    # one product or four: another order of sums, one rounding of the projection (2^-8 in bf16)
        assert a.shape == b.shape and a.dtype == b.dtype and a.requires_grad == b.requires_grad
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() <= (1e-2 if dt == torch.bfloat16 else 1e-5)
    assert len(seen) == 2 * (case == "hook")


def test_prologue_on_projections_refuses():
    modules = [torch.nn.Linear(128, n, bias=False).cuda().bfloat16() for n in (256, 128, 128, 128)]
    x = torch.randn(2, 50, 128, device="cuda").bfloat16().requires_grad_()
    inv = 10000.0 ** (-torch.arange(0, 64, 2, device="cuda").float() / 64)
    for bad in (inv[:16], inv.cpu(), torch.cat([inv, inv])):
        with pytest.raises((ValueError, RuntimeError)):
            _front_call(modules, x, bad)
    with pytest.raises(ValueError):
        _front_call(modules, x, inv, cu=torch.tensor([0, 30, 100], dtype=torch.int32, device="cuda"))
    with pytest.raises(NotImplementedError):
        _front_call(modules, x, inv, fmap="t2r")
