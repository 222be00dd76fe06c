"""Gate gradients: the sums of a chunk's later chunks by the last pass itself, and by a scan over the sequence (taken where
the final states have gradients; zero ones change nothing)."""
import numpy as np
import pytest
import torch

from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu


# (1024 chunks of two heads are the longest sequence whose chunks add up the later ones themselves: one below, one beyond)
@pytest.mark.parametrize("lens,shift", [((1,), 0), ((64, 65), 0), ((16 * 64, 17 * 64), 5), ((33 * 64 + 7, 30, 31 * 64), 64), ((1024 * 64,), 0), ((1024 * 64 + 1,), 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_sum_over_later_chunks_is_the_scan(lens, shift, dtype):
    from nha_amd.ops import nha_prefill, nha_prefill_bwd
    from tests.test_gpu_prefill import KEYS
    cu = np.cumsum((0, *lens)).astype(np.int32)
    T, N, HQ, H, D = int(cu[-1]), len(lens), 4, 2, 64
    d = prefill_inputs(T, 1, T, HQ, H, D, D, 64, dtype=dtype, qk_scale=0.5)
    xs = [d[k][0].cuda().contiguous() for k in KEYS]
    kw = dict(wl=31, shift=shift, scale=D ** -0.5)
    o, lw, lg, _, _ = nha_prefill(*xs, cu, **kw)
    do = torch.randn(T, HQ, D, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
    zero = tuple(torch.zeros(N, H, 64, 64, device="cuda") for _ in range(2))
    a = nha_prefill_bwd(*xs, o, lw, lg, do, cu, **kw)
    b = nha_prefill_bwd(*xs, o, lw, lg, do, cu, dht=zero, **kw)
    for i in range(7):
        if i != 6:
            assert torch.equal(a[i], b[i])
    x, y = a[6].double(), b[6].double()
    if N == 1 and (T + 63) // 64 > 1024:      # both by the scan
        assert torch.equal(x, y)
    # two orders of up to 34 fp32 sums (of the longest sequence's chunks, if more) whose terms are no larger than twice the largest
    # result, then each side's rounding to the dtype (half a unit in the last place: 2^-8 of the value in bf16, 2^-24 in fp32)
    sums = max(34, -(-max(lens) // 64))
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    bound = 2 * sums * 2.0 ** -24 * 2 * y.abs().amax() + 2 * half * torch.maximum(x.abs(), y.abs())
    assert ((x - y).abs() <= bound).all()
    assert x.abs().sum() > 0 or T <= shift


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_infinite_sum_of_a_later_chunk(dtype):
    """The gate gradients of a sequence's last chunk add up to more than float32 holds: those before are infinite, not NaN."""
    from nha_amd.ops import nha_prefill, nha_prefill_bwd
    cu = np.array([0, 192], np.int32)
    T, H, D, M = 192, 2, 64, 64
    one = torch.ones(T, H, D, dtype=dtype, device="cuda")
    strength = torch.zeros(T, H, M, dtype=dtype, device="cuda")
    strength[..., 0] = 1
    xs = [one] * 5 + [strength, torch.zeros_like(strength)]
    kw = dict(wl=31, shift=0, scale=1.0)
    o, lw, lg, _, _ = nha_prefill(*xs, cu, **kw)
    # slot 0 alone is written and read: its logit is 64 (t + 1) in row t, exact in every step, with the cotangent c = 2^111, and dg of row r is
    # 64 c r (T - r): 3e37 at the last row, 1.4e39 at the first of the last chunk (row 128), 1.1e39 at row 48, whose own chunk adds
    # -2.5e38 to the infinite sum (from rows further up it would be -inf)
    dl = torch.full((T, H), 2.0 ** 111, device="cuda")
    zero = tuple(torch.zeros(1, H, 64, 64, device="cuda") for _ in range(2))
    a, b = (nha_prefill_bwd(*xs, o, lw, lg, torch.zeros_like(o), cu, dlse_gsa=dl, dht=dht, **kw)[6][..., 0].float() for dht in (None, zero))
    assert (b[48:129] == torch.inf).all() and b[188:].isfinite().all()
    assert (a[48:129] == torch.inf).all() and torch.equal(a[188:], b[188:])
