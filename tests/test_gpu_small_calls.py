"""Rules that pick a split by the size of the call, on both sides of each line: key groups of the window's dk / dv (64 per
workgroup below, 128 or 256 above), against the fp32 kernels, which share no code with them.  The bf16 kernels see the same rounded inputs, so the tolerances are those of the parity tests:
outputs 2e-2 absolute + 1e-2 relative per element, gradients 1e-2 relative L2 (two or three bf16 roundings of 2^-9 each).
dg is a reverse cumulative sum over the sequence whose terms carry independent roundings while the sum itself stays as
large as the few rows the gates remember: its error grows with the square root of the length, from the 1e-2 that the
340-token cases of the backward's parity tests are held to."""
import pytest
import torch

from tests.test_gpu_prefill_bwd import check_grad
from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
KEYS = ["q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g"]


# 132 key groups of 256 or 110 of 128 for 48 / 12 heads of 128
@pytest.mark.parametrize("D,T,wl", [(128, 2800, 300), (128, 2800, 130), (128, 1200, 130), (128, 1000, 300), (256, 2800, 300), (64, 2800, 100)])
def test_backward_groups(D, T, wl):
    from nha_amd import chunk_nha
    H, NG = 12, 4
    d = prefill_inputs(9100 + D + T + wl, 1, T, H * NG, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5)
    do = torch.randn(1, T, H * NG, D, generator=torch.Generator().manual_seed(3)).to(BF).cuda()
    x = [d[k].cuda().requires_grad_() for k in KEYS]
    grads = torch.autograd.grad(chunk_nha(*x, window_size_left=wl)[0], x, do)
    for h in (0, H - 1):                                   # kv-heads share nothing: two of them, in fp32
        part = [t.detach()[:, :, (NG * h if t.shape[2] > H else h):(NG * (h + 1) if t.shape[2] > H else h + 1)] for t in x]
        ref_in = [t.float().contiguous().requires_grad_() for t in part]
        ro = chunk_nha(*ref_in, window_size_left=wl)[0]
        ref = torch.autograd.grad(ro, ref_in, do[:, :, NG * h:NG * (h + 1)].float())
        for k, g, r in zip(KEYS, grads, ref):
            n = NG if g.shape[2] > H else 1
            check_grad(f"d{k} D{D} T{T} wl{wl} kv-head {h}", g[:, :, n * h:n * (h + 1)], r.cpu(), BF,
                       rel_bar=1e-2 * max(1.0, (T / 340) ** 0.5) if k == "g" else 1e-2)
