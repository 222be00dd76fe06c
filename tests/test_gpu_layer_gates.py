"""The layer prologue's gates over every bf16 logit, four and eight to a lane, against the chain of bf16 operations in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [1, 4, 5, 8])      # rows of 64, 256 (four logits to a lane), 320 and 512 (eight)
@pytest.mark.parametrize("normalizer", [1.0, 8.0])
def test_gates_of_every_bf16_logit(H, normalizer):
    from nha_amd.ops import nha_layer_prologue
    M, K = 64, 16
    bits = torch.arange(65536, dtype=torch.int32).to(torch.uint16).view(torch.bfloat16)
    f = bits[~bits.isnan()]
    T = -(-f.numel() // (H * M))
    f = torch.cat([f, f.new_zeros(T * H * M - f.numel())]).view(1, T, H, M).cuda()
    z = lambda h, d: torch.zeros(1, T, h, d, dtype=torch.bfloat16, device="cuda")
    leaf = f.clone().requires_grad_()
    out = nha_layer_prologue(z(H, K), z(H, K), z(H, K), leaf, torch.ones(K // 2, device="cuda"), feature_map="swish",
                             gate_logit_normalizer=normalizer)
    s, g = out[5].detach().double(), out[6].detach().double()
    r = lambda x: x.to(torch.bfloat16).double()
    x = f.double()
    want_g = r(r(x.clamp(max=0) - torch.log1p(torch.exp(-x.abs()))) / normalizer)
    want_s = r(1 - r(torch.exp(want_g)))
    # fp32 within 3 units in the last place of the true value before each rounding: another bf16 number only where the value is
    # that close to the middle of two (3 / 2^15 of all values per rounding, a half of them wrongly); then the next one
    # (results below the smallest normal number, which the hardware's exponential gives as 0, stand apart)
    for got, want in ((g, want_g), (s, r(1 - r(torch.exp(g))))):
        off = (got != want) & ~((want.abs() < 2.0 ** -120) & (got.abs() < 2.0 ** -120))
        assert off.double().mean() < 1e-3
        assert ((got - want).abs()[off] <= 2.0 ** -7 * want.abs()[off]).all()
    assert torch.equal(g.isinf(), want_g.isinf()) and not g.isnan().any() and not s.isnan().any() and (want_s - s).abs().max() <= 2.0 ** -8
    # d g / d f = sigmoid(-f) / normalizer (with ds zero), rounded once
    dg = torch.autograd.grad(out[6], leaf, torch.ones_like(out[6]))[0].double()
    want = torch.sigmoid(-x) / normalizer
    ok = want > 2.0 ** -120
    assert ((dg - want).abs()[ok] <= 2.0 ** -8 * 1.01 * want[ok]).all()


@pytest.mark.parametrize("H", [4, 8])
@pytest.mark.parametrize("normalizer", [1.0, 8.0, 16.0, 0.5, 3.0, -1.0])
def test_gates_are_the_rounded_values(H, normalizer):
    """Every bf16 logit, subnormal results and NaN included: the values of the 64-bit chain, each step rounded to bf16 once."""
    from nha_amd.ops import nha_layer_prologue
    M, K = 64, 16
    f = torch.arange(65536, dtype=torch.int32).to(torch.uint16).view(torch.bfloat16).view(1, -1, H, M).cuda()
    z = torch.zeros(1, f.shape[1], H, K, dtype=torch.bfloat16, device="cuda")
    out = nha_layer_prologue(z, z, z, f, torch.ones(K // 2, device="cuda"), feature_map="swish", gate_logit_normalizer=normalizer)
    s, g = out[5].double(), out[6].double()
    r = lambda x: x.to(torch.bfloat16).double()
    x = f.double()
    want = r(r(x.clamp(max=0) - torch.log1p(torch.exp(-x.abs()))) / normalizer)
    same = lambda a, b: torch.equal(a.nan_to_num(7.0, torch.inf, -torch.inf), b.nan_to_num(7.0, torch.inf, -torch.inf))
    assert same(g, want) and torch.equal(g.isnan(), x.isnan())
    assert same(s, r(1 - r(torch.exp(g)))) and torch.equal(s.isnan(), x.isnan())
