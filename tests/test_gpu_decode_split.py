"""The decode step of few (sequence, kv-head) pairs (decode_split.hip) against the ring recurrence of the oracle: pairs
around the edges of its dispatch (1, an uneven number, 64, 128, 256 and more), windows of one task, of fewer and of more
32-key blocks than the workgroups have waves, empty, partly filled and wrapped rings, and three steps on one scratch (the
arrival counters must be zero again after each)."""
import pytest
import torch

from oracle import nha_ref as R
from tests.util import assert_close, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,NG,H,K,W", [(1, 8, 1, 128, 33), (1, 4, 2, 128, 700), (3, 3, 3, 64, 64), (2, 1, 2, 256, 300),
                                        (3, 2, 3, 256, 40), (16, 4, 4, 128, 130), (43, 5, 3, 64, 150), (64, 8, 2, 128, 96),
                                        (70, 4, 4, 128, 65), (130, 2, 2, 128, 48)])
def test_split_ring_steps(B, NG, H, K, W):
    from nha_amd import NHARingState, ring_decode_step
    dtype, HQ, M = torch.bfloat16, NG * H, 64
    gen = torch.Generator().manual_seed(B * W + K)
    ring = [randn(gen, B, W, H, d, dtype=dtype) for d in (K, K, K)]
    ring.append((torch.nn.functional.logsigmoid(torch.randn(B, W, H, M, generator=gen)) / 8).to(dtype))
    hk, hv = randn(gen, B, H, K, M, dtype=torch.float32, scale=0.3), randn(gen, B, H, M, K, dtype=torch.float32, scale=0.3)
    count = torch.randint(0, 3 * W, (B,), generator=gen, dtype=torch.int32)
    count[0] = 0 if B > 1 else 2 * W + 5
    count[-1] = W
    st = NHARingState(*[x.clone().cuda() for x in (hk, hv, *ring, count)])
    for i in range(3):
        new = [randn(gen, B, h, K, dtype=dtype) for h in (HQ, HQ, H, H, H)]
        g = (torch.nn.functional.logsigmoid(torch.randn(B, H, M, generator=gen)) / 8).to(dtype)
        o = ring_decode_step(st, *[x.cuda() for x in (*new, g)])
        ro, hk, hv, ring = R.decode_ring_ref(*new, g, *ring, count, hk, hv)
        count = count + 1
        assert_close(f"step {i} o", o, ro, dtype)
        assert_close(f"step {i} hk", st.hk, hk, dtype)
        assert_close(f"step {i} hv", st.hv, hv, dtype)
        assert torch.equal(st.count.cpu(), count)
        for a, b in zip((st.ring_k, st.ring_kg, st.ring_v, st.ring_g), ring):
            assert torch.equal(a.cpu().double(), b)
    from nha_amd import ops
    assert not any(ws[:512].any() for ws in ops._DECODE_SCRATCH.values())      # the counters the next step starts from


def test_split_step_in_a_graph_without_scratch_of_its_own():
    """The window form recorded into a graph on fresh scratch, replayed with eager steps in between: every replay equals
    the eager result (the arrival counters of a recording are its own)."""
    from nha_amd import fused_recurrent_nha_decode
    B, HQ, H, K, W, M, dt = 2, 8, 2, 128, 200, 64, torch.bfloat16
    gen = torch.Generator().manual_seed(3)
    r = lambda *s: randn(gen, *s, dtype=dt).cuda()
    a = dict(q=r(B, 1, HQ, K), sq=r(B, 1, HQ, K), k=r(B, 1, H, K), v=r(B, 1, H, K), g=-r(B, 1, H, M).abs() / 8, sw_k=r(B, W, H, K),
             sw_v=r(B, W, H, K), initial_state=(r(B, H, K, M).float(), r(B, H, M, K).float()), output_final_state=True)
    want, (whk, whv) = fused_recurrent_nha_decode(**a)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        o, (hk, hv) = fused_recurrent_nha_decode(**a)
    for _ in range(4):
        o.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want) and torch.equal(hk, whk) and torch.equal(hv, whv)
        assert torch.equal(fused_recurrent_nha_decode(**a)[0], want)


@pytest.mark.parametrize("B,NG,H,K,W", [(1, 4, 2, 128, 200), (3, 2, 1, 256, 40), (2, 8, 2, 64, 20), (40, 4, 4, 128, 64)])
@pytest.mark.parametrize("where", ["q", "sq", "slots of one task", "keys of one task", "values"])
def test_split_step_keeps_nan(B, NG, H, K, W, where):
    """NaN in all that one part of a pair's work sees reaches the pair's output (the part's maximum does not carry it), and
    no other pair's."""
    from nha_amd import NHARingState, ring_decode_step
    dt, HQ, M, nan = torch.bfloat16, NG * H, 64, float("nan")
    gen = torch.Generator().manual_seed(W)
    ring = [randn(gen, B, W, H, d, dtype=dt) for d in (K, K, K)] + [-randn(gen, B, W, H, M, dtype=dt).abs()]
    hk, hv = randn(gen, B, H, K, M, dtype=torch.float32), randn(gen, B, H, M, K, dtype=torch.float32)
    new = [randn(gen, B, h, K, dtype=dt) for h in (HQ, HQ, H, H, H)] + [-randn(gen, B, H, M, dtype=dt).abs()]
    count = torch.full((B,), 2 * W, dtype=torch.int32)
    if where == "q":
        new[0][0, 0] = nan
    elif where == "sq":
        new[1][0, 0] = nan
    elif where == "slots of one task":
        hk[0, 0, :, 8:16] = nan
    elif where == "keys of one task":
        ring[0][0, :32, 0] = nan
        new[2][0, 0] = nan
    else:
        ring[2][0, W // 2, 0] = nan
    want = R.decode_ring_ref(*new, *ring, count, hk, hv)[0]
    st = NHARingState(*[x.clone().cuda() for x in (hk, hv, *ring, count)])
    o = ring_decode_step(st, *[x.cuda() for x in new]).cpu()
    assert want.isnan().any() and torch.equal(o.isnan(), want.isnan())


def test_split_step_with_a_task_of_slots_that_weigh_nothing():
    """The eight slots of one task at logit -inf: their weight is 0, the rest of the softmax stands."""
    from nha_amd import NHARingState, ring_decode_step
    B, HQ, H, K, W, M, dt = 2, 4, 1, 128, 100, 64, torch.bfloat16
    gen = torch.Generator().manual_seed(5)
    ring = [randn(gen, B, W, H, d, dtype=dt) for d in (K, K, K)] + [-randn(gen, B, W, H, M, dtype=dt).abs()]
    hk, hv = randn(gen, B, H, K, M, dtype=torch.float32), randn(gen, B, H, M, K, dtype=torch.float32)
    hk[..., 16:24] = -float("inf")
    new = [randn(gen, B, h, K, dtype=dt) for h in (HQ, HQ, H, H, H)] + [-randn(gen, B, H, M, dtype=dt).abs()]
    new[0] = new[0].abs() + 0.01
    count = torch.full((B,), 2 * W, dtype=torch.int32)
    want = R.decode_ring_ref(*new, *ring, count, hk, hv)[0]
    st = NHARingState(*[x.clone().cuda() for x in (hk, hv, *ring, count)])
    assert_close("o", ring_decode_step(st, *[x.cuda() for x in new]), want, dt)


def test_split_steps_on_more_streams_than_scratch_is_kept_for():
    """Four threads, each taking the window form through new streams of its own: 24 in all, more than the pool keeps."""
    import threading
    from nha_amd import fused_recurrent_nha_decode, ops
    B, HQ, H, K, W, M, dt = 2, 8, 2, 128, 200, 64, torch.bfloat16
    gen = torch.Generator().manual_seed(9)
    r = lambda *s: randn(gen, *s, dtype=dt).cuda()
    a = dict(q=r(B, 1, HQ, K), sq=r(B, 1, HQ, K), k=r(B, 1, H, K), v=r(B, 1, H, K), g=-r(B, 1, H, M).abs() / 8, sw_k=r(B, W, H, K),
             sw_v=r(B, W, H, K), initial_state=(r(B, H, K, M).float(), r(B, H, M, K).float()), output_final_state=True)
    want = fused_recurrent_nha_decode(**a)[0]
    torch.cuda.synchronize()
    got, streams = [], [[torch.cuda.Stream() for _ in range(6)] for _ in range(4)]

    def work(mine):
        for s in mine:
            with torch.cuda.stream(s):
                for _ in range(5):
                    o = fused_recurrent_nha_decode(**a)[0]
                s.synchronize()
                got.append(torch.equal(o, want))
    threads = [threading.Thread(target=work, args=(x,)) for x in streams]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert got == [True] * 24 and len(ops._DECODE_SCRATCH) <= ops._WORKSPACE_MAX_STREAMS


# pairs that are split, that keep one workgroup of four waves, and that keep the kernel of large calls
@pytest.mark.parametrize("B,NG,H,K,W", [(3, 4, 2, 128, 200), (3, 8, 1, 64, 33), (2, 1, 2, 256, 300), (80, 4, 4, 128, 64), (3, 3, 64, 64, 40),
                                        (160, 4, 4, 64, 48)])
@pytest.mark.parametrize("value", ["nan", "inf"])
def test_ring_rows_without_a_token_are_not_looked_at(B, NG, H, K, W, value):
    """A ring that is not full pops nothing: rows past its count may hold anything (fresh memory, an earlier request's), and
    the step is that of a ring with zeros there."""
    from nha_amd import NHARingState, ring_decode_step
    dt, HQ, M = torch.bfloat16, NG * H, 64
    gen = torch.Generator().manual_seed(W + B)
    clean = [randn(gen, B, W, H, d, dtype=dt) for d in (K, K, K)] + [-randn(gen, B, W, H, M, dtype=dt).abs()]
    hk, hv = randn(gen, B, H, K, M, dtype=torch.float32, scale=0.3), randn(gen, B, H, M, K, dtype=torch.float32, scale=0.3)
    count = torch.tensor([0, 1, W - 1] * B, dtype=torch.int32)[:B]
    empty = (torch.arange(W)[None] >= count[:, None])[..., None, None]
    clean = [x.masked_fill(empty, 0) for x in clean]
    st = NHARingState(*[x.clone().cuda() for x in (hk, hv, *[x.masked_fill(empty, float(value)) for x in clean], count)])
    new = [randn(gen, B, h, K, dtype=dt) for h in (HQ, HQ, H, H, H)] + [-randn(gen, B, H, M, dtype=dt).abs()]
    o = ring_decode_step(st, *[x.cuda() for x in new])
    ro, hk, hv, ring = R.decode_ring_ref(*new, *clean, count, hk, hv)
    for name, a, b in (("o", o, ro), ("hk", st.hk, hk), ("hv", st.hv, hv)):
        assert_close(name, a, b, dt)


@pytest.mark.parametrize("name", ["q", "k", "v", "g", "s"])
def test_window_step_on_operands_off_a_16_byte_boundary(name):
    """A contiguous view one element into its buffer goes to the kernel that reads single elements: the output is its, bit for
    bit, at a size that is split otherwise."""
    from nha_amd import fused_recurrent_nha_decode, ops
    B, HQ, H, K, W, M, dt = 2, 8, 2, 128, 200, 64, torch.bfloat16
    gen = torch.Generator().manual_seed(4)
    r = lambda *s: randn(gen, *s, dtype=dt).cuda()
    a = dict(q=r(B, 1, HQ, K), sq=r(B, 1, HQ, K), k=r(B, 1, H, K), v=r(B, 1, H, K), g=-r(B, 1, H, M).abs() / 8, s=r(B, 1, H, M).abs(),
             sw_k=r(B, W, H, K), sw_v=r(B, W, H, K), initial_state=(r(B, H, K, M).float(), r(B, H, M, K).float()), output_final_state=True)
    o, state = fused_recurrent_nha_decode(**a)
    small = torch.zeros(16, dtype=torch.uint8, device="cuda")
    keep, ops.decode_scratch = ops.decode_scratch, lambda dev, stream: small      # too small to be split over workgroups
    try:
        unsplit, want = fused_recurrent_nha_decode(**a)
    finally:
        ops.decode_scratch = keep
    assert not torch.equal(state[0], want[0]) or not torch.equal(o, unsplit)      # two kernels, two orders of sums
    x = a[name]
    a[name] = torch.empty(x.numel() + 1, dtype=dt, device="cuda")[1:].view(x.shape).copy_(x)
    assert a[name].is_contiguous() and a[name].data_ptr() % 16
    got, (hk, hv) = fused_recurrent_nha_decode(**a)
    assert torch.equal(got, unsplit) and torch.equal(hk, want[0]) and torch.equal(hv, want[1])


@pytest.mark.parametrize("B,W,fills", [(3, 200, 1), (130, 64, 0)])
def test_recorded_steps_take_scratch_where_they_use_it(B, W, fills, monkeypatch):
    """A recording makes (and so fills, at every replay) scratch for the steps that use it only; its replays are the eager step."""
    from nha_amd import NHARingState, ops, ring_decode_step
    HQ, H, K, M, dt = 8, 2, 128, 64, torch.bfloat16
    gen = torch.Generator().manual_seed(W)
    r = lambda *s: randn(gen, *s, dtype=dt).cuda()
    first = [randn(gen, B, H, *s, dtype=torch.float32, scale=0.3).cuda() for s in ((K, M), (M, K))] + [r(B, W, H, K) for _ in range(3)] + \
        [-r(B, W, H, M).abs(), torch.full((B,), 2 * W + 1, dtype=torch.int32, device="cuda")]
    new = [r(B, HQ, K), r(B, HQ, K), r(B, H, K), r(B, H, K), r(B, H, K), -r(B, H, M).abs()]
    eager = NHARingState(*[x.clone() for x in first])
    want = ring_decode_step(eager, *new, advance=False)
    st, made, make = NHARingState(*[x.clone() for x in first]), [], ops.new_decode_scratch
    monkeypatch.setattr(ops, "new_decode_scratch", lambda dev: made.append(1) or make(dev))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        o = ring_decode_step(st, *new, advance=False)
    assert len(made) == fills
    for _ in range(3):
        for x, y in zip((st.hk, st.hv, st.ring_k, st.ring_kg, st.ring_v, st.ring_g), first):
            x.copy_(y)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want) and torch.equal(st.hk, eager.hk) and torch.equal(st.ring_v, eager.ring_v)
