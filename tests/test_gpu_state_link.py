"""The second level of the forward's state pass as one launch, which adds up the end states before each segment (bf16 path), against
the fp32-math kernels, which know no segments: gates that never decay, so that every segment of a sequence reaches all later ones;
gates whose decay is zero within a segment; growing ones; sequences of one chunk beside long ones, an odd number of segments before
one, with and without states.  Tolerances of the parity tests (2e-2 absolute + 1e-2 relative per element)."""
import numpy as np
import pytest
import torch

from tests.util import assert_close, prefill_inputs

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
KEYS = ["q_swa", "k_swa", "q_gsa", "k_gsa", "v", "s", "g"]


@pytest.mark.parametrize("gates", ["none", "fast", "growing", "mixed"])
@pytest.mark.parametrize("states", [False, True])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_linked_segments(D, states, gates):
    from nha_amd import chunk_nha
    H, lens = 2, [1500, 64, 1, 700, 130]
    cu = torch.tensor([0, *np.cumsum(lens).tolist()], dtype=torch.int32, device="cuda")
    d = prefill_inputs(9700 + D, 1, sum(lens), H, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5, with_state=states, N=len(lens))
    c = {k: d[k].cuda() for k in KEYS}
    c["s"] = c["s"] * 0.02                            # what the slots take up without decay stays of the order of one
    if gates == "none":
        c["g"].zero_()
    elif gates == "fast":
        c["g"].fill_(-3.0)                            # e^-192 per chunk
    elif gates == "growing":
        c["g"] = (c["g"] / -200).clamp(0, 0.001)
    else:
        c["g"][..., ::3] = 0
        c["g"][..., 1::3] = -3.0
    kw = dict(cu_seqlens=cu, window_size_left=70, gsa_kv_shift=71, output_final_state=True)
    if states:
        kw["initial_state"] = tuple(t.cuda() for t in d["h0"])
    got = chunk_nha(*c.values(), **kw)
    ref = chunk_nha(*(x.float() for x in c.values()), impl="simple", **kw)
    for name, x, y in zip(("o", "lse_swa", "lse_gsa", "hk", "hv"), (*got[:3], *got[3]), (*ref[:3], *ref[3])):
        assert_close(f"{name} D{D} states{states} {gates}", x, y, BF)


def _with_one_odd_value(D, lens, where, value, gates):
    """Operands (two kv-heads), initial states and options of a call with one infinity or NaN: in token 10 of the first sequence, or in
    its initial state."""
    H = 2
    d = prefill_inputs(9800 + D, 1, sum(lens), H, H, D, D, 64, dtype=BF, qk_scale=D ** -0.5, with_state=True, N=len(lens), gate_div=gates)
    c, h0 = {k: d[k].cuda() for k in KEYS}, [t.cuda() for t in d["h0"]]
    if where in ("hk", "hv"):
        h0["hk hv".split().index(where)][0, 1, 5, 6] = value
    else:
        c[where][0, 10, 1, 6] = value
    cu = torch.tensor([0, *np.cumsum(lens).tolist()], dtype=torch.int32, device="cuda")
    return c, dict(cu_seqlens=cu, window_size_left=63, gsa_kv_shift=64, output_final_state=True, initial_state=tuple(h0))


LINKED, SCANNED = [1500, 64, 1, 700, 130], [3000]     # sequences whose second level is one launch; a scan and a rewrite
ODD = [("v", float("nan")), ("k_gsa", float("inf")), ("s", float("nan")), ("hk", float("nan")), ("hv", float("-inf"))]


@pytest.mark.parametrize("where,value", ODD)
@pytest.mark.parametrize("gates", [8.0, 1.0])          # decays that are zero in fp32 after some 150 and some 1000 tokens
@pytest.mark.parametrize("D,lens", [(64, LINKED), (128, LINKED), (256, LINKED), (128, SCANNED), (256, SCANNED)])
def test_infinities_and_nans_reach_the_final_state(D, lens, gates, where, value):
    """Whatever the gates forget: the same elements of the final states are not finite as token by token (fp32 kernels)."""
    from nha_amd import chunk_nha
    c, kw = _with_one_odd_value(D, lens, where, value, gates)
    got, ref = chunk_nha(*c.values(), **kw)[3], chunk_nha(*(x.float() for x in c.values()), impl="simple", **kw)[3]
    assert any((~y.isfinite()).any() for y in ref)
    for name, x, y in zip(("hk", "hv"), got, ref):
        assert torch.equal(x.isfinite(), y.isfinite()), name
