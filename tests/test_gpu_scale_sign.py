"""Scales below and at zero: every output pass and window gradient of the matrix cores against the generic fp32 kernels on the same
bf16-rounded inputs."""
import pytest
import torch

from tests.test_gpu_prefill_bwd import BF, KEYS, check_grad
from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,NG,D", [(16, 1, 64), (4, 2, 64), (2, 4, 64), (4, 1, 128), (4, 2, 128), (2, 3, 128), (2, 4, 128), (4, 1, 256)])
@pytest.mark.parametrize("sign", [-1.0, 0.0])
@pytest.mark.parametrize("wl", [64, -1])
def test_forward_and_gradients(H, NG, D, sign, wl):
    from nha_amd import chunk_nha
    print("case", H, NG, D, sign, wl, flush=True)
    cu = torch.tensor([0, 1, 40, 104, 361], dtype=torch.int32).cuda()
    d = prefill_inputs(77 + D + NG, 1, 361, H * NG, H, D, D, 64, dtype=BF)
    do = torch.randn(1, 361, H * NG, D, generator=torch.Generator().manual_seed(3)).to(BF)
    res = []
    for dt, impl in ((BF, "mfma"), (torch.float32, "simple")):
        x = [d[k].cuda().to(dt).requires_grad_(True) for k in KEYS]
        out = chunk_nha(*x, cu_seqlens=cu, scale=sign * D ** -0.5, window_size_left=wl, gsa_kv_shift=16, impl=impl)
        res.append([*(t.detach() for t in out), *torch.autograd.grad(out[0], x, do.cuda().to(dt))])
    for name, got, ref in zip(("o", "lse_swa", "lse_gsa", *("d" + k for k in KEYS)), *res):
        check_grad(name, got, ref.double().cpu(), BF)


@pytest.mark.parametrize("HQ,H,D,T", [(8, 2, 128, 95), (16, 4, 64, 300), (72, 18, 128, 500)])   # two heads a workgroup, two, four
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_broken_window_queries_at_a_scale_of_zero(HQ, H, D, T, value):
    """0 times an infinity or a NaN is a NaN: the query's own output row is not finite, and no other (fp32 kernels)."""
    from nha_amd import chunk_nha
    d = prefill_inputs(78, 1, T, HQ, H, D, D, 64, dtype=BF)
    d["q_swa"][0, 70, 3, 5] = value
    got, ref = (chunk_nha(*(d[k].cuda().to(dt) for k in KEYS), scale=0.0, window_size_left=63, impl=impl)[0].isfinite()
                for dt, impl in ((BF, "mfma"), (torch.float32, "simple")))
    assert not ref[0, 70, 3].any() and ref.sum().item() == ref.numel() - D
    assert (got != ref).sum().item() == 0
