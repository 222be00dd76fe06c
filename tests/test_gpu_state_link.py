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
