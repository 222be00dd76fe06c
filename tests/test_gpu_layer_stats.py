"""The epilogue's backward with a wave per row (dim <= 2048) at the edges of its columns and row groups, and the slot
branch's share of the softmax mass, against the fp64 formulas."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


# one row; a ragged group; dims at the edges of 512 columns per step and of 1024 (eight waves or four); many groups
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,dim", [(1, 8), (9, 512), (45, 520), (8192, 64), (8195, 1024), (61, 1032), (70, 2048), (8225, 1544)])
def test_epilogue_backward_rows(dtype, rows, dim):
    from nha_amd.ops import nha_layer_epilogue
    gen = torch.Generator().manual_seed(rows + dim)
    o, dy = ((2 * torch.randn(rows, dim, generator=gen)).to(dtype) for _ in range(2))
    w, b = 1 + 0.3 * torch.randn(dim, generator=gen), torch.randn(dim, generator=gen)
    x = [o.cuda().requires_grad_(), w.cuda().requires_grad_(), b.cuda().requires_grad_()]
    got = torch.autograd.grad(nha_layer_epilogue(*x, 1e-5), x, dy.cuda())
    y = [t.double().requires_grad_() for t in (o, w, b)]
    a = F.silu(y[0])
    n = a * torch.rsqrt(a.pow(2).mean(-1, keepdim=True) + 1e-5)
    ref = torch.autograd.grad(n * y[1] + y[2], y, dy.double())
    # bf16: silu(o) and do are rounded (2^-9 each); fp32: sums of dim or rows terms
    bar = 1e-2 if dtype == torch.bfloat16 else 1e-5
    for name, g, r in zip(("do", "dweight", "dbias"), got, ref):
        rel = ((g.double().cpu() - r).norm() / r.norm()).item()
        assert rel <= bar, f"{name}: relative L2 error {rel:.3e}"


@pytest.mark.parametrize("n", [1, 255, 65536, 300001])
def test_gsa_share(n):
    from nha_amd.ops import gsa_share
    gen = torch.Generator().manual_seed(n)
    a, b = 30 * torch.randn(n, generator=gen), 30 * torch.randn(n, generator=gen)
    if n > 1:
        a[0], b[1] = float("-inf"), float("-inf")
    ref = torch.sigmoid(b.double() - a.double()).mean().item()
    assert abs(gsa_share(a.cuda(), b.cuda()) - ref) <= 1e-5      # fp32 exponentials and sums of up to 1200 terms
