"""The one-launch hand-over of a prompt to a decode ring against the rule it implements, row by row."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,lens,K,dtype", [
    (1, (1, 2), 64, torch.bfloat16),                  # a ring of one slot
    (16, (1, 15, 16, 17, 33), 8, torch.bfloat16),     # shorter than, equal to and past the window; rows of one piece
    (64, (63, 200), 128, torch.float32),
    (300, (5, 299), 256, torch.bfloat16),             # no prompt fills the ring
    (48, (50, 50, 50), 64, torch.bfloat16),           # equal lengths: also without cu_seqlens
    (16, (20, 7), 3, torch.bfloat16),                 # rows that are not whole 16-byte pieces
])
def test_ring_slots_hold_the_newest_tokens(W, lens, K, dtype):
    from nha_amd import NHARingState
    H, M, N, total = 2, 64, len(lens), sum(lens)
    gen = torch.Generator().manual_seed(W)
    rows = [torch.randn(1, total, H, d, generator=gen).to(dtype) for d in (K, K, K, M)]
    states = [torch.randn(N, H, K, M, generator=gen), torch.randn(N, H, M, K, generator=gen)]
    cu = [0, *itertools.accumulate(lens)]
    want = [torch.zeros(N, W, H, x.shape[-1], dtype=dtype) for x in rows]
    for n, L in enumerate(lens):
        for j in range(max(0, L - W), L):
            for ring, x in zip(want, rows):
                ring[n, j % W] = x[0, cu[n] + j]
    dev = [x.cuda() for x in rows]
    calls = [(dev, torch.tensor(cu, dtype=torch.int32).cuda()), (dev, torch.tensor(cu)),
             ([x.transpose(1, 2).contiguous().transpose(1, 2) for x in dev], torch.tensor(cu).cuda())]   # another order in memory
    if len(set(lens)) == 1:
        calls.append(([x.reshape(N, lens[0], *x.shape[2:]) for x in dev], None))
    for ops, bounds in calls:
        sd = [x.cuda() for x in states]
        st = NHARingState.from_prefill(*ops, tuple(sd), W, cu_seqlens=bounds)
        assert st.count.dtype == torch.int32 and st.count.tolist() == list(lens)
        for got, ref in zip((st.ring_k, st.ring_kg, st.ring_v, st.ring_g), want):
            assert torch.equal(got.cpu(), ref)
        assert torch.equal(st.hk.cpu(), states[0]) and torch.equal(st.hv.cpu(), states[1])
        assert st.hk.data_ptr() != sd[0].data_ptr()     # a copy: the caller's states stay the caller's
