"""The one-launch slot branch of the bf16 backward (prefill_bwd_slot.hip) against reverse-mode differentiation of the fp64
recurrence, at the places where its tiling can go wrong.

Tolerances are those of test_gpu_prefill_bwd.py: o, do and the gradients are bf16 (2^-9 = 2e-3 per rounding), and a gradient
sums products of two or three such roundings with independent signs, so 1e-2 in relative L2; tables made from fp32
intermediates are kept to 16 bits of mantissa and add nothing to that."""
import pytest
import torch

from tests.test_gpu_prefill_bwd import BF, run_bwd_case
from tests.util import prefill_inputs

pytestmark = pytest.mark.gpu

# one row, the last row of the first half, the first of the second, a whole chunk, one row of a second chunk, three chunks
CU = [0, 1, 33, 66, 130, 195, 340]


@pytest.mark.parametrize("shift", [0, 32, 70])
@pytest.mark.parametrize("NG", [1, 3])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_slot_branch_edges(D, NG, shift):
    """Ragged chunks, one and several query heads per kv-head, sequences shorter than the shift, a shift past a chunk."""
    H = 2
    d = prefill_inputs(8100 + D + NG + shift, 1, CU[-1], H * NG, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5, with_state=True, N=len(CU) - 1)
    run_bwd_case(f"slot D{D} NG{NG} shift{shift}", d, wl=40, shift=shift, dtype=BF, cu=CU, with_dht=True)


@pytest.mark.parametrize("gate_mean", [-2.0, -5.0])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_slot_branch_strong_gates(D, gate_mean):
    """Chunks whose decay leaves the factored form's range (about e^-70 within a half at -2: some chunks; all at -5) are
    taken by the launch that forms the decay pair by pair; the LSE's own cotangent included."""
    d = prefill_inputs(8200 + D, 1, CU[-1], 4, 2, D, D, 64, dtype=BF, qk_scale=D ** -0.5, gate_div=1.0, gate_mean=gate_mean,
                       with_state=True, N=len(CU) - 1)
    run_bwd_case(f"slot strong {gate_mean} D{D}", d, wl=40, shift=0, dtype=BF, cu=CU, with_lse=True)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_slot_branch_growing_gates_beside_strong_ones(D):
    """Slots that grow (log gates up to +0.01) in chunks that others make strongly decaying: the decay of a pair is formed as it
    is, above 1 too."""
    d = prefill_inputs(8300 + D, 1, CU[-1], 4, 2, D, D, 64, dtype=BF, qk_scale=D ** -0.5, gate_div=1.0, gate_mean=-5.0,
                       with_state=True, N=len(CU) - 1)
    d["g"][..., 8:] = (d["g"][..., 8:] / -400).clamp(0, 0.01)
    d["s"][..., 8:] = (d["s"][..., 8:] / 20)
    run_bwd_case(f"slot growing D{D}", d, wl=40, shift=0, dtype=BF, cu=CU, with_lse=True)


@pytest.mark.parametrize("gate_mean", [0.0, -2.0])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_slot_branch_one_head_per_kv_head(D, gate_mean):
    """One query head per kv-head has an instance of its own (all columns in one workgroup, nothing summed over heads): an odd
    number of heads, the LSE's own cotangent, and at -2 chunks that are left to the launch for strongly decaying ones."""
    d = prefill_inputs(8400 + D, 1, CU[-1], 3, 3, D, D, 64, dtype=BF, qk_scale=D ** -0.5, gate_div=1.0, gate_mean=gate_mean,
                       with_state=True, N=len(CU) - 1)
    run_bwd_case(f"slot one head {gate_mean} D{D}", d, wl=40, shift=33, dtype=BF, cu=CU, with_lse=True)


@pytest.mark.parametrize("gate_mean", [0.0, -2.0])
@pytest.mark.parametrize("NG", [4, 6, 8])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_slot_branch_heads_in_parts(D, NG, gate_mean):
    """Few chunks and kv-heads: a kv-head's query heads are shared out over 4, 2 and 8 workgroups (six heads: three to each of two),
    whose sums the scan over the chunks adds up; a shift that leaves tokens without a row, and at -2 chunks of the launch for
    strongly decaying ones.  The bound of dg is that of the strong gates with final states (test_gpu_prefill_bwd.py): their
    cotangents enter it at every token with terms that cancel, and all heads summed in one workgroup give the same 0.9 to 1.12e-2."""
    d = prefill_inputs(8500 + D + NG, 1, CU[-1], 2 * NG, 2, D, D, 64, dtype=BF, qk_scale=D ** -0.5, gate_div=1.0, gate_mean=gate_mean,
                       with_state=True, N=len(CU) - 1)
    run_bwd_case(f"slot parts {gate_mean} D{D} NG{NG}", d, wl=40, shift=33, dtype=BF, cu=CU, with_dht=True, dg_bar=2e-2)
