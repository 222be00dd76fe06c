"""Window gradients from the LDS-direct kernels (K = V = 128: a multiple of four query heads per kv-head; K = V =
256: any grouping, more than 256 chunks x kv-heads or query heads to share out, few empty halves of 128-row workgroups) against the fp32 call (generic
kernels) on the same bf16-rounded inputs: ragged packed sequences that end inside a 32-row unit, a chunk and a group of chunks,
windows below and above those where the kernels and their key groups change, odd and even numbers of units, longer than every
sequence and unbounded."""
import pytest
import torch

from tests.test_gpu_prefill_bwd import BF, KEYS, check_grad
from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu


def compare(cu, wl, H, NG, D, keys, scale=None, shift=0):
    from nha_amd import chunk_nha
    d = prefill_inputs(9100 + wl + NG, 1, cu[-1], H * NG, H, D, D, 64, dtype=BF, qk_scale=1.0)
    do = torch.randn(1, cu[-1], H * NG, D, generator=torch.Generator().manual_seed(wl + 5)).to(BF)
    outs, grads = [], []
    for dt in (BF, torch.float32):
        x = [d[k].cuda().to(dt).requires_grad_(True) for k in KEYS]
        o = chunk_nha(*x, cu_seqlens=torch.tensor(cu, dtype=torch.int32).cuda(),
                      scale=D ** -0.5 if scale is None else scale, window_size_left=wl, gsa_kv_shift=shift)[0]
        o.backward(do.cuda().to(dt))
        outs.append(o.detach())
        grads.append([t.grad for t in x])
    check_grad(f"wl={wl} o", outs[0], outs[1].double().cpu(), BF)
    for k, gb, gf in zip(KEYS, *grads):
        if k in keys:
            check_grad(f"wl={wl} d{k}", gb, gf.double().cpu(), BF)


# 1, 1, 1, 5 and 13 chunks: seven in eight halves of 128-row workgroups are taken as filled (too few for some of the 256-wide kernels); 1, 1, 1, 5
# and 12, four on average: all
CU, CU256 = [0, 1, 40, 104, 361, 1190], [0, 1, 40, 104, 361, 1126]


@pytest.mark.parametrize("H,NG,D,cu", [(32, 4, 128, CU), (32, 8, 128, CU), (16, 1, 256, CU), (13, 3, 256, CU), (16, 1, 256, CU256), (13, 3, 256, CU256)])
@pytest.mark.parametrize("wl", [-1, 0, 31, 64, 159, 160, 192, 383, 384, 500, 2000])
def test_window_gradients_of_many_key_groups(wl, H, NG, D, cu):
    print("case", wl, H, NG, D, flush=True)
    # otherwise other kernels take dk and dv
    chunks = sum((b - a + 63) // 64 for a, b in zip(cu, cu[1:]))
    assert H * chunks > 256 if D == 256 else H * (chunks // 4) > 128
    compare(cu, wl, H, NG, D, ("q_swa", "k_swa", "v"))


@pytest.mark.parametrize("H,NG,D", [(24, 2, 64), (25, 2, 64), (12, 3, 128), (13, 3, 128), (5, 1, 128), (6, 2, 256), (7, 2, 256)])
@pytest.mark.parametrize("wl", [-1, 0, 64, 159])
def test_window_gradients_of_few_key_groups(wl, H, NG, D):
    """dk and dv of 64 keys by four or by eight waves: the last sizes of the one and the first of the other (21 groups of keys per
    kv-head), tiles of 64 queries whose second half is empty, and ends inside either half."""
    print("case", wl, H, NG, D, flush=True)
    compare(CU, wl, H, NG, D, ("k_swa", "v"))


@pytest.mark.parametrize("H,NG", [(11, 4), (12, 8), (13, 4), (23, 4), (24, 4), (43, 4)])
@pytest.mark.parametrize("wl", [-1, 160, 192, 500])
def test_window_gradients_of_128_keys_in_two_groups(wl, H, NG):
    """Head size 128, 11 groups of 128 keys and 6 of 256 per kv-head: the last size without (11) and the first and last (12, 23; 43) with two
    groups of waves on 128 keys; units alone and with their complements, an odd number of them, items of fewer queries than 32."""
    print("case", wl, H, NG, flush=True)
    compare(CU, wl, H, NG, 128, ("k_swa", "v"))


@pytest.mark.parametrize("H,NG,D", [(10, 4, 128), (9, 4, 128), (4, 12, 128), (2, 8, 128), (1, 4, 128), (10, 2, 256), (3, 6, 256), (5, 4, 256), (2, 8, 256)])
@pytest.mark.parametrize("wl", [-1, 40, 159, 160, 300])
def test_window_gradients_of_query_heads_in_parts(wl, H, NG, D):
    """Few groups of 128 keys: a kv-head's query heads are shared out over 2, 4 (three heads to each of four at 12) and 8 workgroups whose
    fp32 sums the last pass of the gates adds up; (10, 4, 128) is the first size without.  A shift that leaves the last tokens of a
    sequence, and whole sequences, without a slot part of dv."""
    print("case", wl, H, NG, D, flush=True)
    compare(CU256 if D == 256 else CU, wl, H, NG, D, ("k_swa", "v", "q_swa"), shift=50)


@pytest.mark.parametrize("wl", [40, 400])
def test_more_sequences_than_lanes(wl):
    """150 ragged sequences of up to 130 tokens, empty ones among them: the forward's workgroups of two chunks search among them, the
    window gradients fall to kernels of 64 rows."""
    lens = [(37 * i) % 131 for i in range(150)]
    cu = torch.tensor([0, *lens]).cumsum(0).tolist()
    print("case", wl, flush=True)
    compare(cu, wl, 4, 1, 256, KEYS)


@pytest.mark.parametrize("N,H", [(64, 4), (68, 4), (152, 4), (4100, 1)])
@pytest.mark.parametrize("wl", [40, 400])
def test_pairs_of_many_sequences(wl, N, H):
    """The workgroups of two chunks count the pairs of up to 64 sequences and search among more, in steps of 64 and of 4096: one to three chunks
    each, two on average (taken as filled; the 256-wide window gradients of others fall to kernels of 64 rows), empty ones among them."""
    lens = [(65, 1, 130, 66)[i % 4] for i in range(N)]
    lens[N // 2:N // 2] = [0, 0]
    cu = torch.tensor([0, *lens]).cumsum(0).tolist()
    print("case", wl, N, H, flush=True)
    compare(cu, wl, H, 1, 256, KEYS)


@pytest.mark.parametrize("H,NG,D,cu", [(32, 4, 128, CU), (16, 1, 256, CU), (16, 1, 256, CU256)])
@pytest.mark.parametrize("wl", [-1, 64, 200, 500])
def test_negative_scale(wl, H, NG, D, cu):
    """The weights of the keys outside the window are zero whatever the sign of the scale."""
    print("case", wl, H, NG, D, flush=True)
    compare(cu, wl, H, NG, D, KEYS, scale=-D ** -0.5)


@pytest.mark.parametrize("scale", [0.0, 1e-42, -1e-42, 1e-28])
@pytest.mark.parametrize("wl", [64, 500])
def test_scale_of_zero(wl, scale):
    """All keys of the window weigh the same; dk_swa is zero, or nearly so, and finite."""
    print("case", wl, scale, flush=True)
    compare(CU, wl, 32, 4, 128, ("k_swa", "v"), scale=scale)


@pytest.mark.parametrize("H,NG,D,dt", [(32, 4, 128, BF), (2, 4, 128, BF), (16, 1, 256, BF), (2, 1, 256, BF), (4, 1, 64, BF), (4, 1, 64, torch.float32)])
@pytest.mark.parametrize("wl", [2**31 - 1, 2**31 - 1000, 2**30])
def test_longest_windows_are_unbounded(wl, H, NG, D, dt):
    from nha_amd import chunk_nha
    print("case", wl, H, NG, D, dt, flush=True)
    cu = torch.tensor(CU256, dtype=torch.int32).cuda()
    d = prefill_inputs(5, 1, CU256[-1], H * NG, H, D, D, 64, dtype=dt)
    do = torch.randn(1, CU256[-1], H * NG, D, generator=torch.Generator().manual_seed(2)).to(dt).cuda()
    res = []
    for w in (-1, wl):
        x = [d[k].cuda().requires_grad_(True) for k in KEYS]
        out = chunk_nha(*x, cu_seqlens=cu, window_size_left=w, gsa_kv_shift=0)
        res.append([*out, *torch.autograd.grad(out[0], x, do)])
    assert all(torch.equal(p, q) for p, q in zip(*res))
