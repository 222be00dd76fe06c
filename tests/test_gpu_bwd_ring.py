"""Window gradients from the LDS-direct kernels (four or eight query heads per kv-head at K = V = 128, more key groups than 128)
against the fp32 call (generic kernels) on the same bf16-rounded inputs: ragged packed sequences that end inside a 32-row unit,
a chunk and a group of four chunks, windows below and above the 160 keys where the key groups change size, odd and even numbers
of units, longer than every sequence and unbounded."""
import pytest
import torch

from tests.test_gpu_prefill_bwd import BF, KEYS, check_grad
from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NG", [4, 8])
@pytest.mark.parametrize("wl", [-1, 0, 31, 64, 159, 160, 383, 500, 2000])
def test_window_gradients_of_many_key_groups(wl, NG):
    from nha_amd import chunk_nha
    H, D, M = 32, 128, 64
    cu = [0, 1, 40, 104, 361, 1190]
    print("case", wl, NG, flush=True)
    assert H * (sum((b - a + 63) // 64 for a, b in zip(cu, cu[1:])) // 4) > 128     # otherwise other kernels take dk and dv
    d = prefill_inputs(9100 + wl + NG, 1, cu[-1], H * NG, H, D, D, M, dtype=BF, qk_scale=1.0)
    do = torch.randn(1, cu[-1], H * NG, D, generator=torch.Generator().manual_seed(wl + 5)).to(BF)
    grads = []
    for dt in (BF, torch.float32):
        x = [d[k].cuda().to(dt).requires_grad_(True) for k in KEYS]
        o = chunk_nha(*x, cu_seqlens=torch.tensor(cu, dtype=torch.int32).cuda(), scale=D ** -0.5, window_size_left=wl, gsa_kv_shift=0)[0]
        o.backward(do.cuda().to(dt))
        grads.append([t.grad for t in x])
    for k, gb, gf in zip(KEYS, *grads):
        if k in ("q_swa", "k_swa", "v"):
            check_grad(f"wl={wl} d{k}", gb, gf.double().cpu(), BF)
