"""Rules that pick a split by the size of the call, on both sides of each line: chunks per segment of the bf16 state pass
(1 to 8), key groups of the window's dk / dv (64 per workgroup below, 128 or 256 above), where the output pass keeps its
decay fragments; against the fp32 kernels, which share no code with them.  The bf16 kernels see the same rounded inputs, so
the tolerances are those of the parity tests:
outputs 2e-2 absolute + 1e-2 relative per element, gradients 1e-2 relative L2 (two or three bf16 roundings of 2^-9 each).
dg is a reverse cumulative sum over the sequence whose terms carry independent roundings while the sum itself stays as
large as the few rows the gates remember: its error grows with the square root of the length, from the 1e-2 that the
340-token cases of the backward's parity tests are held to."""
import numpy as np
import pytest
import torch

from tests.test_gpu_prefill_bwd import check_grad
from tests.util import assert_close, prefill_inputs

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
KEYS = ["q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g"]


# chunks per segment: 1, 2, 4, 8 (long chains), 8 (a full chip), mixed lengths with 1 and with 4
@pytest.mark.parametrize("D,H,lens", [(128, 2, [450]), (64, 1, [1500]), (128, 2, [6000]), (128, 1, [16500]), (256, 12, [1500, 1300]),
                                      (256, 2, [1, 65, 129, 64, 700]), (64, 16, [17, 1000, 64, 130, 1700])])
@pytest.mark.parametrize("shift", [0, 96])
def test_segment_lengths(D, H, lens, shift):
    from nha_amd import chunk_nha
    cu = torch.tensor([0, *np.cumsum(lens).tolist()], dtype=torch.int32, device="cuda")
    d = prefill_inputs(9000 + D + H, 1, sum(lens), H, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5, with_state=True, N=len(lens))
    c = [d[k].cuda() for k in KEYS]
    h0 = tuple(t.cuda() for t in d["h0"])
    kw = dict(cu_seqlens=cu, window_size_left=70, gsa_kv_shift=shift, initial_state=h0, output_final_state=True)
    o, ls, lg, st = chunk_nha(*c, **kw)
    ro, rls, rlg, rst = chunk_nha(*(x.float() for x in c), impl="simple", **kw)
    for name, x, y in (("o", o, ro), ("lse_swa", ls, rls), ("lse_gsa", lg, rlg), ("hk", st[0], rst[0]), ("hv", st[1], rst[1])):
        assert_close(f"{name} D{D} H{H} {lens} shift{shift}", x, y, BF)


# 132 key groups of 256 or 110 of 128 for 48 / 12 heads of 128; segments of 4, 8 and 2 chunks in the backward's state pass
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


# two query heads per kv-head: 224 and 264 workgroups of the output pass, either side of the 256 CUs
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [1786, 2100])
def test_output_pass_pairs(D, T):
    from nha_amd import chunk_nha
    H = 8
    d = prefill_inputs(9200 + D + T, 1, T, 2 * H, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5, gate_div=1.0, gate_mean=-1.0)
    c = [d[k].cuda() for k in KEYS]
    got = chunk_nha(*c, window_size_left=150)
    ref = chunk_nha(*(x.float() for x in c), window_size_left=150, impl="simple")
    for name, x, y in zip(("o", "lse_swa", "lse_gsa"), got, ref):
        assert_close(f"{name} D{D} T{T}", x, y, BF)
