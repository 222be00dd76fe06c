"""The fp32 matrix-core prefill (prefill_f32.hip) against the fp64 oracle: head sizes, groupings, lengths around the
16-row and 64-row edges, sequences shorter than the shift, unbounded windows, initial states, and gates that forget by more
than e^-60 within 16 rows (the pairwise decay form), everywhere or in single slots."""
import numpy as np
import pytest
import torch

from tests.test_gpu_prefill import run_case
from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu
F32 = torch.float32


@pytest.mark.parametrize("D,HQ,H", [(64, 4, 4), (64, 10, 2), (128, 8, 2), (128, 3, 1), (256, 2, 1)])
@pytest.mark.parametrize("T,wl,shift", [(15, 3, 0), (17, 16, 17), (64, 63, 64), (65, 0, 1), (200, 15, 16), (333, 100, 0), (150, -1, 3)])
def test_f32_edges(D, HQ, H, T, wl, shift):
    d = prefill_inputs(T * D + HQ, 2, T, HQ, H, D, D, 64, dtype=F32, qk_scale=0.5, with_state=T % 2 == 1)
    run_case(f"D{D} {HQ}/{H} T{T} wl{wl} shift{shift}", d, wl=wl, shift=shift, dtype=F32, impl=None)


@pytest.mark.parametrize("lens,wl,shift", [((1, 200, 3, 50, 4, 130, 2, 7), 31, 32), ((128, 64, 70, 10), 40, 0), ((300, 1, 129), 200, 70)])
def test_f32_varlen(lens, wl, shift):
    cu = [0] + np.cumsum(lens).tolist()
    d = prefill_inputs(len(lens), 1, cu[-1], 4, 2, 64, 64, 64, dtype=F32, with_state=True, N=len(lens))
    run_case(f"varlen {lens}", d, wl=wl, shift=shift, dtype=F32, impl=None, cu=cu)


@pytest.mark.parametrize("mean", [-4.0, -8.0])
def test_f32_strong_gates(mean):
    """16 rows forget by up to e^-130 (mean -8): growing decay factors would pass the fp32 range.  Then single fast slots."""
    d = prefill_inputs(7, 1, 150, 4, 2, 64, 64, 64, dtype=F32, gate_div=1.0, gate_mean=mean, with_state=True)
    run_case(f"gates {mean}", d, wl=20, shift=0, dtype=F32, impl=None)
    d = prefill_inputs(8, 1, 150, 4, 2, 128, 128, 64, dtype=F32)
    d["g"][:, 40:75, :, 5] = mean
    d["s"] = 1 - d["g"].exp()
    run_case(f"one fast slot {mean}", d, wl=20, shift=5, dtype=F32, impl=None)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("name", ["q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g", "h0k", "h0v"])
def test_f32_nan_reaches_every_output_that_depends_on_it(name, D):
    """NaN in one row of an operand: every output that is NaN in the recurrence is NaN here (a maximum or a clamp drops
    NaN where it is not looked after), and tokens of the 16-row blocks before it are untouched."""
    from nha_amd import chunk_nha
    from oracle import nha_ref as R
    from tests.test_gpu_prefill import KEYS
    at, T, wl = 70, 200, 20
    d = prefill_inputs(D, 1, T, 4, 2, D, D, 64, dtype=F32, with_state=True)
    if name in ("h0k", "h0v"):
        d["h0"][name == "h0v"][:, 1, 3] = float("nan")
        at = 0
    else:
        d[name][:, at] = float("nan")
    ref = R.prefill_ref(*[d[k] for k in KEYS], window_size_left=wl, gsa_kv_shift=0, initial_state=d["h0"])
    o, lse_swa, lse_gsa, (hkt, hvt) = chunk_nha(*[d[k].cuda() for k in KEYS], window_size_left=wl, window_size_right=0,
                                                initial_state=tuple(x.cuda() for x in d["h0"]), output_final_state=True)
    assert any(x.isnan().any() for x in ref)
    for what, got, want in zip(("o", "lse_swa", "lse_gsa", "hk", "hv"), (o, lse_swa, lse_gsa, hkt, hvt), ref):
        got, want = got.cpu(), want.reshape(got.shape)
        assert not (want.isnan() & ~got.isnan()).any(), what
        if what in ("o", "lse_swa", "lse_gsa"):
            assert got[:, :at // 16 * 16].isfinite().all(), what


@pytest.mark.parametrize("T,D,div,mean", [(512, 64, 1.0, 0.0), (700, 256, 8.0, 0.0), (896, 128, 1.0, -1.0)])
def test_f32_states_are_no_less_exact_than_the_generic_kernels(T, D, div, mean):
    """Error of the final states against 64 bits, beside that of the generic kernels: decays formed from cumsums rounded at
    the chunk's magnitude were 1.2 times theirs; a quarter of an fp32 rounding is left for the order of the sums."""
    from nha_amd import chunk_nha
    from oracle import nha_ref as R
    from tests.test_gpu_prefill import KEYS
    d = prefill_inputs(1, 1, T, 4, 4, D, D, 64, dtype=F32, gate_div=div, gate_mean=mean, qk_scale=D ** -0.5, with_state=True)
    ref = R.prefill_ref(*[d[k] for k in KEYS], window_size_left=63, gsa_kv_shift=0, initial_state=d["h0"])[3:]
    errs = {}
    for impl in ("simple", None):
        got = chunk_nha(*[d[k].cuda() for k in KEYS], window_size_left=63, window_size_right=0, impl=impl,
                        initial_state=tuple(x.cuda() for x in d["h0"]), output_final_state=True)[3]
        errs[impl] = [((a.double().cpu() - b).norm() / b.norm()).item() for a, b in zip(got, ref)]
    print(errs)
    assert all(a <= b + 2.0 ** -26 for a, b in zip(errs[None], errs["simple"])), errs


# (window, shift): slots that absorb every token at once, the window's hand-over, a gap between window and slots (the last
# `shift` tokens are absorbed by nobody; the one at 195 is one of them)
@pytest.mark.parametrize("D,wl,shift", [(64, 20, 0), (128, 19, 20), (64, 5, 37), (256, 20, 0)])
@pytest.mark.parametrize("at", [70, 111, 195])
@pytest.mark.parametrize("name,value", [(n, "nan") for n in ("q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g")] +
                         [(n, "inf") for n in ("k_swa", "k_gsa", "v", "s")])
def test_f32_rows_that_a_token_does_not_see(name, value, at, D, wl, shift):
    """A row that is not finite reaches exactly the outputs that depend on it: not earlier tokens of its 16-row block, nor
    tokens that it has left the window of, nor, where no slot has absorbed it, any later one.  (The products take 16 rows at
    once, the unseen ones with weight zero, and zero times NaN or inf is NaN.)"""
    from nha_amd import chunk_nha
    from oracle import nha_ref as R
    from tests.test_gpu_prefill import KEYS
    from tests.util import assert_close
    d = prefill_inputs(D + at, 1, 200, 4, 2, D, D, 64, dtype=F32, qk_scale=0.5, with_state=True)
    d[name][:, at, 1, :] = float(value)
    ref = R.prefill_ref(*[d[k] for k in KEYS], window_size_left=wl, gsa_kv_shift=shift, initial_state=d["h0"])
    o, lse_swa, lse_gsa, (hkt, hvt) = chunk_nha(*[d[k].cuda() for k in KEYS], window_size_left=wl, window_size_right=0, gsa_kv_shift=shift,
                                                initial_state=tuple(x.cuda() for x in d["h0"]), output_final_state=True)
    assert any(not x.isfinite().all() for x in ref) or at == 195
    for what, got, want in zip(("o", "lse_swa", "lse_gsa", "hk", "hv"), (o, lse_swa, lse_gsa, hkt, hvt), ref):
        got, want = got.cpu(), want.reshape(got.shape)
        assert torch.equal(got.isfinite(), want.isfinite()), (what, got.isfinite().sum().item(), want.isfinite().sum().item())
        assert_close(what, got.masked_fill(~got.isfinite(), 0), want.masked_fill(~want.isfinite(), 0), F32)


@pytest.mark.parametrize("name", ["q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g", "h0k", "h0v"])
def test_f32_operands_off_a_16_byte_boundary(name):
    """A contiguous view one float into its buffer: the matrix-core kernels, which read 16 bytes at a time, leave the call to
    the generic ones wherever they would read it so."""
    from nha_amd import chunk_nha
    from tests.test_gpu_prefill import KEYS
    d = prefill_inputs(3, 1, 90, 4, 2, 64, 64, 64, dtype=F32, qk_scale=0.5, with_state=True)
    c = {k: x.cuda() for k, x in d.items() if k in KEYS}
    c["h0k"], c["h0v"] = (x.cuda() for x in d["h0"])
    buf = torch.empty(c[name].numel() + 1, dtype=F32, device="cuda")
    call = lambda impl: chunk_nha(*[c[k] for k in KEYS], window_size_left=20, window_size_right=0, impl=impl,
                                  initial_state=(c["h0k"], c["h0v"]), output_final_state=True)
    flat = lambda out: [*out[:3], *out[3]]
    fast, want = flat(call(None)), flat(call("simple"))
    assert not torch.equal(fast[0], want[0])              # two kernels, two orders of sums
    c[name] = buf[1:].view(c[name].shape).copy_(c[name])
    assert c[name].is_contiguous() and c[name].data_ptr() % 16
    if name in ("g", "h0k"):                              # single floats in both
        want = fast
    assert all(torch.equal(x, y) for x, y in zip(flat(call(None)), want))


@pytest.mark.parametrize("T,D,HQ,H,wl,shift,mean", [(1, 64, 4, 4, 0, 0, 0.0), (17, 64, 6, 2, 63, 64, 0.0), (200, 64, 4, 4, -1, 16, -8.0),
                                                    (79, 128, 5, 1, 16, 0, 0.0), (145, 256, 2, 2, 100, 3, -4.0)])
@pytest.mark.parametrize("bad", [None, "v", "k_swa", "s"])
def test_f32_four_waves_or_one_per_unit(T, D, HQ, H, wl, shift, mean, bad):
    """A sequence alone (units of 16 rows and a head below 512: four waves each) and the same one many times over (one wave
    each), against the oracle; with a row of NaN in `bad`, the outputs that are finite in the recurrence are finite."""
    from nha_amd import chunk_nha
    from oracle import nha_ref as R
    from tests.test_gpu_prefill import KEYS
    from tests.util import assert_close
    d = prefill_inputs(T + D, 1, T, HQ, H, D, D, 64, dtype=F32, qk_scale=0.5, gate_div=1.0, gate_mean=mean, with_state=True)
    if bad:
        d[bad][:, T // 2] = float("nan")
    ref = R.prefill_ref(*[d[k] for k in KEYS], window_size_left=wl, gsa_kv_shift=shift, initial_state=d["h0"])[:3]
    units = (T + 63) // 64 * 4 * HQ
    for B in (1, 512 // units + 1):
        assert (B * units <= 512) == (B == 1)
        out = chunk_nha(*[d[k].cuda().expand(B, -1, -1, -1) for k in KEYS], window_size_left=wl, window_size_right=0, gsa_kv_shift=shift,
                        initial_state=tuple(x.cuda().expand(B, -1, -1, -1) for x in d["h0"]))
        for what, got, want in zip(("o", "lse_swa", "lse_gsa"), out, ref):
            assert torch.equal(got.nan_to_num(7.0), got[:1].nan_to_num(7.0).expand_as(got))      # every copy the same
            got, want = got[:1].cpu(), want.reshape(got[:1].shape)
            assert torch.equal(got.isfinite(), want.isfinite()), (what, B)
            assert_close(what, got.masked_fill(~got.isfinite(), 0), want.masked_fill(~want.isfinite(), 0), F32)
