"""GPU parity of the bf16 MFMA prefill kernels against the fp64 oracle (small/medium shapes) and
against the independent fp32-math HIP kernels (larger shapes), through the C ABI."""
import itertools
import random

import numpy as np
import pytest
import torch

from oracle import nha_ref as R
from tests.test_gpu_prefill import KEYS, run_case
from tests.util import assert_close, prefill_inputs

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def test_mfma_reference_grid():
    """The reference's prefill grid shapes that the MFMA kernels serve (M = 64)."""
    seed = 3100
    for T, B, W in itertools.product((63, 128, 257, 1000), (1, 4), (32, 64)):
        d = prefill_inputs(seed, B, T, 8, 2, 64, 64, 64, dtype=BF, with_state=(T == 128))
        seed += 1
        run_case(f"mfma_t{T}_b{B}_w{W} shifted", d, wl=W - 1, shift=W, dtype=BF, impl="mfma")
        if B == 1:
            run_case(f"mfma_t{T}_b{B}_w{W} layer", d, wl=W, shift=0, dtype=BF, impl="mfma")


@pytest.mark.parametrize("D,NG", [(128, 4), (128, 1), (128, 2), (128, 8), (64, 1), (64, 3), (256, 1), (256, 2), (256, 4)])
def test_mfma_head_shapes_and_windows(D, NG):
    H = 2
    for li, (T, wl, shift) in enumerate([(200, 99, 100), (333, 100, 0), (130, -1, 0), (260, 255, 256), (70, 500, 0),
                                         (192, 63, 0), (192, 64, 64), (150, 0, 1)]):
        d = prefill_inputs(500 + 10 * D + NG + li, 2, T, H * NG, H, D, D, 64, dtype=BF, with_state=(li % 2 == 0))
        run_case(f"mfma D{D} NG{NG} T{T} wl{wl} sh{shift}", d, wl=wl, shift=shift, dtype=BF, impl="mfma")


def test_mfma_varlen():
    random.seed(1)
    for li, lens in enumerate([[128, 64, 200, 10], [300, 1, 129, 2, 64], [random.randint(1, 100) for _ in range(40)],
                               [1, 200, 3, 50, 4, 130, 2, 7]]):
        cu = [0] + list(np.cumsum(lens))
        T, H, NG, D = cu[-1], 2, 4, 128
        d = prefill_inputs(700 + li, 1, T, H * NG, H, D, D, 64, dtype=BF, with_state=True, N=len(lens))
        run_case(f"mfma varlen{li} shifted", d, wl=31, shift=32, dtype=BF, impl="mfma", cu=cu)
        run_case(f"mfma varlen{li} layer", d, wl=100, shift=0, dtype=BF, impl="mfma", cu=cu)


def test_mfma_varlen_d256():
    """Scaled-down version of the varlen benchmark config: H=4, D=256, M=64, W=512, random lengths,
    per-sequence initial state ~ N(0, 0.1)."""
    rng = np.random.default_rng(3)
    lens = [int(x) for x in rng.integers(64, 700, size=6)] + [1, 65]
    cu = [0] + list(np.cumsum(lens))
    d = prefill_inputs(750, 1, cu[-1], 4, 4, 256, 256, 64, dtype=BF, with_state=True, N=len(lens), state_scale=0.1,
                       qk_scale=256 ** -0.5, gate_div=1.0)
    run_case("varlen d256 layer", d, wl=512, shift=0, dtype=BF, impl="mfma", cu=cu)
    run_case("varlen d256 shifted", d, wl=511, shift=512, dtype=BF, impl="mfma", cu=cu)


@pytest.mark.parametrize("NG", [1, 2])
def test_mfma_d256_sequences_of_every_chunk_count(NG):
    """The head-size-256 output pass gives a workgroup two consecutive chunks of a sequence: sequences of one to five
    chunks with full and partial last chunks (a lone last chunk, a second chunk of one row), short and long windows,
    slot-branch shifts inside and beyond a chunk, per-sequence initial states, against the fp64 oracle."""
    lens = [1, 64, 65, 128, 129, 191, 192, 257, 320, 17]
    cu = [0] + list(np.cumsum(lens))
    d = prefill_inputs(760 + NG, 1, cu[-1], 2 * NG, 2, 256, 256, 64, dtype=BF, with_state=True, N=len(lens), state_scale=0.1,
                       qk_scale=256 ** -0.5, gate_div=1.0)
    for wl, shift in ((0, 0), (31, 32), (64, 0), (100, 65), (200, 201), (-1, 0)):
        run_case(f"d256 chunk pairs NG{NG} wl{wl} shift{shift}", d, wl=wl, shift=shift, dtype=BF, impl="mfma", cu=cu)
    # mostly single-chunk sequences: the launch with one chunk per workgroup
    lens = [1, 64, 30, 17, 64, 65, 40]
    cu = [0] + list(np.cumsum(lens))
    d = prefill_inputs(770 + NG, 1, cu[-1], 2 * NG, 2, 256, 256, 64, dtype=BF, with_state=True, N=len(lens), state_scale=0.1,
                       qk_scale=256 ** -0.5, gate_div=1.0)
    for wl, shift in ((31, 32), (100, 0)):
        run_case(f"d256 single chunks NG{NG} wl{wl} shift{shift}", d, wl=wl, shift=shift, dtype=BF, impl="mfma", cu=cu)


def test_mfma_slow_forgetting_gates():
    """Gate logits ~ N(-1,1) -> logsigmoid with no /8 normaliser (the long-context config's
    distribution): sum of g over a 16-row sub-block is about -22."""
    d = prefill_inputs(800, 2, 400, 8, 2, 128, 128, 64, dtype=BF, gate_div=1.0, gate_mean=-1.0, qk_scale=128 ** -0.5)
    run_case("slow-forgetting", d, wl=127, shift=128, dtype=BF, impl="mfma")
    run_case("slow-forgetting layer", d, wl=128, shift=0, dtype=BF, impl="mfma")


@pytest.mark.parametrize("gate_mean", [-3.0, -4.5, -6.0, -8.0, -12.0])
def test_mfma_fast_forgetting_gates(gate_mean):
    """Strong forgetting: gate logits ~ N(gate_mean, 1) -> logsigmoid, so a 16-row sub-block decays
    by about e^-50 ... e^-190 and a chunk by far more than fp32 can hold.  Up to e^-80 per sub-block
    the matrix-core slot branch factors the decay exactly; beyond that the state pass flags the
    sub-block and its rows are recomputed with the unfactored decay.  Decayed terms must underflow
    to zero, not to NaN, and the recent rows must stay exact."""
    d = prefill_inputs(850, 2, 300, 8, 2, 128, 128, 64, dtype=BF, gate_div=1.0, gate_mean=gate_mean, qk_scale=128 ** -0.5,
                       with_state=True)
    run_case(f"fast-forgetting {gate_mean}", d, wl=63, shift=64, dtype=BF, impl="mfma")
    run_case(f"fast-forgetting {gate_mean} layer", d, wl=100, shift=0, dtype=BF, impl="mfma")


@pytest.mark.parametrize("D,HQ,H", [(64, 4, 4), (128, 8, 2), (256, 4, 2)])
def test_mfma_isolated_strong_decay(D, HQ, H):
    """A few slots forget abruptly in a few rows of otherwise ordinary, packed sequences: only the
    16-row sub-blocks that contain them take the exact path, everything else the matrix-core path,
    and both must agree with the recurrence."""
    cu = [0, 100, 333, 400]
    d = prefill_inputs(860 + D, 1, cu[-1], HQ, H, D, D, 64, dtype=BF, gate_div=8.0, qk_scale=D ** -0.5, with_state=True,
                       N=3)
    g = d["g"].float()
    g[0, 70:73, 0, 5] = -40.0       # sequence 0, chunk 1, sub-block 0
    g[0, 150, :, 17] = -90.0        # sequence 1 (rows 100..332): row 50 -> chunk 0, sub-block 3
    g[0, 331:333, H - 1, 63] = -60.0   # last rows of sequence 1, ragged chunk
    g[0, 399, 0, :] = -100.0        # the very last row
    d["g"] = g.to(BF)
    run_case("isolated decay layer", d, wl=64, shift=0, dtype=BF, impl="mfma", cu=cu)
    run_case("isolated decay shifted", d, wl=31, shift=32, dtype=BF, impl="mfma", cu=cu)


@pytest.mark.parametrize("HQ,H", [(8, 2), (2, 2)])
@pytest.mark.parametrize("per_row", [-3.55, -4.6])
def test_mfma_decay_near_the_clamp_at_scale_one(HQ, H, per_row):
    """scale = 1 (the layer's default) with q / k of magnitude 2, and slots whose gates decay a 16-row
    sub-block by e^-57 (just inside what the matrix cores factor: s exp(57) times unscaled scores summed
    over 16 rows must stay inside fp32) or by e^-74 (flagged, recomputed exactly).  Logits of this size
    make the softmax sharp, so bf16 rounding of the states moves single outputs by more than the
    element-wise bar: finite everywhere, relative L2 within 3e-2."""
    from nha_amd import chunk_nha
    d = prefill_inputs(870, 2, 192, HQ, H, 64, 64, 64, dtype=BF, gate_div=8.0, qk_scale=2.0)
    g = d["g"].float()
    g[:, 16:32, :, 3] = per_row
    g[:, 80:96, 0, 40:44] = per_row
    g[:, 160:176, H - 1, 63] = per_row
    d["g"] = g.to(BF)
    d["s"] = (1 - d["g"].float().exp()).to(BF)
    for wl, shift in ((31, 32), (64, 0)):
        c = [d[k].cuda() for k in KEYS]
        o, ls, lg = chunk_nha(*c, window_size_left=wl, gsa_kv_shift=shift, scale=1.0, impl="mfma")
        ro, rls, rlg, _, _ = R.prefill_ref(*[d[k] for k in KEYS], window_size_left=wl, gsa_kv_shift=shift, scale=1.0)
        for name, got, ref in (("o", o, ro), ("lse_swa", ls, rls), ("lse_gsa", lg, rlg)):
            got = got.double().cpu()
            assert torch.isfinite(got).all(), name
            rel = ((got - ref).norm() / ref.norm()).item()
            assert rel <= 3e-2, (name, wl, shift, rel)


@pytest.mark.parametrize("HQ,H,D", [(4, 2, 256), (8, 2, 128), (8, 2, 64)])
@pytest.mark.parametrize("qk_scale", [1.0, 3.0])
def test_mfma_scores_far_from_the_fixed_softmax_reference(qk_scale, HQ, H, D):
    """Scale 1 with unnormalised q / k: window scores of a few hundred, far above and far below those of the
    chunk's own keys.  The LDS-direct output passes (four query heads per kv-head at D <= 128, any grouping
    at D = 256) fix the softmax reference of a row from its first keys and hand rows whose sums leave the
    fp32 range they allow (2^+-100 around the reference at D <= 128, 2^96 above it at D = 256) to the exact
    pass.  Finite everywhere, relative L2 within 3e-2 (logits of this size make single outputs move by more
    than the element-wise bar under bf16 rounding of the states)."""
    from nha_amd import chunk_nha
    d = prefill_inputs(880, 2, 200, HQ, H, D, D, 64, dtype=BF, gate_div=8.0, qk_scale=qk_scale)
    for wl, shift in ((99, 100), (64, 0)):
        c = [d[k].cuda() for k in KEYS]
        o, ls, lg = chunk_nha(*c, window_size_left=wl, gsa_kv_shift=shift, scale=1.0, impl="mfma")
        ro, rls, rlg, _, _ = R.prefill_ref(*[d[k] for k in KEYS], window_size_left=wl, gsa_kv_shift=shift, scale=1.0)
        for name, got, ref in (("o", o, ro), ("lse_swa", ls, rls), ("lse_gsa", lg, rlg)):
            got = got.double().cpu()
            assert torch.isfinite(got).all(), (name, wl, shift)
            rel = ((got - ref).norm() / ref.norm()).item()
            assert rel <= 3e-2, (name, wl, shift, rel)


def test_mfma_matches_simple_kernels_at_size():
    """A shape the CPU recurrence cannot reach in seconds: MFMA kernels vs the fp32-math kernels."""
    from nha_amd import chunk_nha
    B, T, HQ, H, D, W = 2, 4096, 8, 2, 128, 1024
    d = prefill_inputs(900, B, T, HQ, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5, gate_div=1.0, gate_mean=-1.0)
    c = [d[k].cuda() for k in KEYS]
    a = chunk_nha(*c, window_size_left=W - 1, gsa_kv_shift=W, output_final_state=True, impl="mfma")
    b = chunk_nha(*c, window_size_left=W - 1, gsa_kv_shift=W, output_final_state=True, impl="simple")
    assert_close("o", a[0], b[0].double(), BF)
    assert_close("lse_swa", a[1], b[1].double(), BF)
    assert_close("lse_gsa", a[2], b[2].double(), BF)
    assert_close("hk", a[3][0], b[3][0].double(), BF)
    assert_close("hv", a[3][1], b[3][1].double(), BF)


@pytest.mark.parametrize("B,T", [(1, 6144), (2, 3072)])
@pytest.mark.parametrize("gate_div,gate_mean", [(8.0, 0.0), (1.0, -1.0)])
def test_mfma_long_sequences_both_forms_of_the_state_carry(B, T, gate_div, gate_mean):
    """Sequences of 24 and 12 segments: the first takes the scan-then-apply form of the state pass's second level, the
    second the form that links the segments itself; with the layers' slow gates (logsigmoid / 8: the carried state reaches every chunk
    of a segment) and with fast ones (everything past a segment's first chunks is left as it is).  Initial states, so
    that the first segment carries something too.  Against the fp32-math kernels."""
    from nha_amd import chunk_nha
    HQ, H, D, W = 8, 2, 128, 256
    d = prefill_inputs(910 + B, B, T, HQ, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5, gate_div=gate_div, gate_mean=gate_mean,
                       with_state=True, state_scale=0.5)
    c = [d[k].cuda() for k in KEYS]
    h0 = (d["h0"][0].cuda(), d["h0"][1].cuda())
    a = chunk_nha(*c, window_size_left=W - 1, gsa_kv_shift=W, initial_state=h0, output_final_state=True, impl="mfma")
    b = chunk_nha(*c, window_size_left=W - 1, gsa_kv_shift=W, initial_state=h0, output_final_state=True, impl="simple")
    assert_close("o", a[0], b[0].double(), BF)
    assert_close("lse_gsa", a[2], b[2].double(), BF)
    assert_close("hk", a[3][0], b[3][0].double(), BF)
    assert_close("hv", a[3][1], b[3][1].double(), BF)
    for nm, x, y in (("o", a[0], b[0]), ("hk", a[3][0], b[3][0]), ("hv", a[3][1], b[3][1])):
        rel = ((x.double() - y.double()).norm() / y.double().norm()).item()
        assert rel <= 5e-3, f"{nm}: relative L2 error {rel:.3e}"


def test_mfma_headline_shape_matches_c_oracle():
    """The benchmark's own shape (T=8192, 32/8 heads, D=128, M=64, W=2048; one of its two sequences)
    element by element against the plain-C restatement of the oracle, which gets through it in
    seconds on the host cores."""
    import bench
    from nha_amd import chunk_nha
    from oracle.nha_ref_c import prefill_ref_c
    cfg = bench.PREFILL
    xs = bench.make_prefill_inputs(torch, cfg, "cpu", seed=5, B=1)
    W = cfg["W"]
    ref = prefill_ref_c(*xs, window_size_left=W - 1, gsa_kv_shift=W)
    got = chunk_nha(*[x.cuda() for x in xs], window_size_left=W - 1, gsa_kv_shift=W, output_final_state=True, impl="mfma")
    assert_close("o", got[0], ref[0].double(), BF)
    assert_close("lse_swa", got[1], ref[1].double(), BF)
    assert_close("lse_gsa", got[2], ref[2].double(), BF)
    assert_close("hk", got[3][0], ref[3].double(), BF)
    assert_close("hv", got[3][1], ref[4].double(), BF)
    # the workload's values are small next to the absolute bar above: relative L2 error as well
    # (bf16 output rounding alone is 2^-9)
    for name, a, b in (("o", got[0], ref[0]), ("hk", got[3][0], ref[3]), ("hv", got[3][1], ref[4])):
        rel = ((a.double().cpu() - b.double()).norm() / b.double().norm()).item()
        assert rel <= 5e-3, f"{name}: relative L2 error {rel:.3e}"


@pytest.mark.parametrize("name", ["cfg2", "cfg3", "cfg5"])
def test_mfma_layer_workloads_match_c_oracle(name):
    """The other configurations, with their own input distributions, against the C restatement:
    cfg2 (340M-layer shape, D=256, layer convention wl = W, shift = 0, gate logits N(0,1), no
    initial state; 2 of its 8 independent sequences), cfg3 (the packed varlen draw of 64..4096-token
    sequences, 32768 tokens, initial states ~ N(0, 0.1)) and cfg5 (32/8 heads, D=128, W=2048,
    gate logits N(-1,1), shifted convention; 1 of its 2 independent T=16384 sequences)."""
    import bench
    from nha_amd import chunk_nha
    from oracle.nha_ref_c import prefill_ref_c
    cfg = dict(bench.WORKLOADS[name])
    if not cfg.get("varlen"):
        cfg["B"] = 1 if name == "cfg5" else 2                 # a part of its batch
    lens = bench.workload_lengths(torch, cfg)
    xs = bench.make_prefill_inputs(torch, cfg, "cpu", seed=9)
    cu = None
    if cfg.get("varlen"):
        cu = torch.tensor([0] + list(itertools.accumulate(lens)), dtype=torch.int32)
    h0 = bench.make_initial_state(torch, cfg, len(lens), "cpu")
    assert (h0 is not None) == (name == "cfg3")
    kw = dict(window_size_left=cfg.get("wl", cfg["W"] - 1), gsa_kv_shift=cfg.get("shift", cfg["W"]))
    ref = prefill_ref_c(*xs, cu_seqlens=None if cu is None else cu.tolist(), initial_state=h0, **kw)
    got = chunk_nha(*[x.cuda() for x in xs], cu_seqlens=None if cu is None else cu.cuda(),
                    initial_state=None if h0 is None else (h0[0].cuda(), h0[1].cuda()), output_final_state=True,
                    impl="mfma", **kw)
    assert_close("o", got[0], ref[0].double(), BF)
    assert_close("lse_swa", got[1], ref[1].double(), BF)
    assert_close("lse_gsa", got[2], ref[2].double(), BF)
    assert_close("hk", got[3][0], ref[3].double(), BF)
    assert_close("hv", got[3][1], ref[4].double(), BF)
    # the absolute bar says little where a tensor's values are small (final states of about 0.05 at these input
    # scales): relative L2 error of every output as well (bf16 output rounding alone is 2^-9)
    for nm, a, b in (("o", got[0], ref[0]), ("lse_swa", got[1], ref[1]), ("lse_gsa", got[2], ref[2]),
                     ("hk", got[3][0], ref[3]), ("hv", got[3][1], ref[4])):
        rel = ((a.double().cpu() - b.double()).norm() / b.double().norm()).item()
        assert rel <= 5e-3, f"{nm}: relative L2 error {rel:.3e}"


@pytest.mark.parametrize("H,NG,D", [(18, 4, 128), (16, 4, 128), (9, 8, 64), (8, 8, 64), (2, 2, 128), (33, 2, 128), (3, 6, 128)])
@pytest.mark.parametrize("scale", [1.0, -1.0, 0.0])
@pytest.mark.parametrize("wl", [-1, 0, 64, 200])
def test_ring_one_and_two_row_blocks_per_wave(H, NG, D, scale, wl):
    """Eight chunks: 72 query heads are the first multiple of four whose workgroups take four heads each, 64 the last with two; two and six
    heads per kv-head are mfma_out_kernel's.  Sequences that end inside a row block, scales of both signs and zero, against the generic fp32
    kernels on the same bf16-rounded inputs: probabilities and outputs rounded to bf16, 1e-2 in relative L2."""
    from nha_amd import chunk_nha
    from tests.test_gpu_prefill_bwd import check_grad
    print("case", H, NG, D, scale, wl, flush=True)
    cu = torch.tensor([0, 1, 40, 104, 361], dtype=torch.int32).cuda()
    d = prefill_inputs(880 + D + NG, 1, 361, H * NG, H, D, D, 64, dtype=BF, with_state=True, N=4)
    h0 = tuple(x.cuda() for x in d["h0"])
    res = [chunk_nha(*(d[k].cuda().to(dt) for k in KEYS), cu_seqlens=cu, scale=scale * D ** -0.5, window_size_left=wl, gsa_kv_shift=16,
                     initial_state=h0, impl=impl)[:3] for dt, impl in ((BF, "mfma"), (torch.float32, "simple"))]
    for name, got, ref in zip(("o", "lse_swa", "lse_gsa"), *res):
        check_grad(name, got, ref.double().cpu(), BF)


@pytest.mark.parametrize("HQ,H,lens,wl", [(8, 4, [700, 700], 64), (8, 4, [300], 128), (12, 2, [900], 200), (8, 4, [1500, 1500], 399)])
def test_strong_logits_of_two_and_six_heads(HQ, H, lens, wl):
    """Window logits of std 4: single keys dominate, and what the fixed softmax reference of the LDS-direct pass leaves to bf16's rounding
    of the probabilities shows.  Relative errors against fp32 over these four calls, mfma_out_kernel / the LDS-direct pass: window
    log-sum-exp 6.0e-5 to 7.1e-5 / 7.7e-5 to 1.06e-4, outputs 1.75e-3 to 2.05e-3 / 1.81e-3 to 2.10e-3; the bounds lie between."""
    from nha_amd import chunk_nha
    cu = torch.tensor([0, *itertools.accumulate(lens)], dtype=torch.int32).cuda()
    bound = 7.0e-5 if lens[0] == 1500 else 7.9e-5
    for seed in range(2):
        d = prefill_inputs(7100 + seed, 1, sum(lens), HQ, H, 128, 128, 64, dtype=BF, qk_scale=2.0)
        got, ref = (chunk_nha(*(d[k].cuda().to(dt) for k in KEYS), cu_seqlens=cu, window_size_left=wl, impl=impl)
                    for dt, impl in ((BF, "mfma"), (torch.float32, "simple")))
        rel = ((got[1] - ref[1]).norm() / ref[1].norm()).item()
        print("log-sum-exp", HQ, H, lens, rel, flush=True)
        assert rel < bound


@pytest.mark.parametrize("HQ,H,D,lens,wl,qk", [(32, 4, 128, [1000], 300, 0.3), (32, 4, 128, [331], 63, 0.3), (16, 4, 64, [331], 63, 0.2)])
def test_small_logits_and_fast_gates_of_small_calls(HQ, H, D, lens, wl, qk):
    """Small calls of four heads per kv-head, window logits around zero, gates that forget within a few tokens: where the softmax
    reference lies decides how finely bf16 holds the probabilities.  Mean relative error of the output against fp32 over four seeds, with a reference
    of 0 / of log2(245/256): 2.307e-3 / 2.339e-3, 2.300e-3 / 2.335e-3, 2.298e-3 / 2.342e-3; the bound lies between."""
    from nha_amd import chunk_nha
    cu = torch.tensor([0, *itertools.accumulate(lens)], dtype=torch.int32).cuda()
    errors = []
    for seed in range(4):
        d = prefill_inputs(7200 + seed, 1, sum(lens), HQ, H, D, D, 64, dtype=BF, gate_div=1.0, gate_mean=-1.0, qk_scale=qk)
        d["v"] = (d["v"].float() / qk).to(BF)
        got, ref = (chunk_nha(*(d[k].cuda().to(dt) for k in KEYS), cu_seqlens=cu, window_size_left=wl, impl=impl)[0].double()
                    for dt, impl in ((BF, "mfma"), (torch.float32, "simple")))
        errors.append(((got - ref).norm() / ref.norm()).item())
    print("output", HQ, H, D, lens, errors, flush=True)
    assert sum(errors) / 4 < 2.32e-3
