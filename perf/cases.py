"""The workloads that the library's speed is judged by: what a user of the operators, the decode cache, the layer and
the hybrid attention blocks has them do, through their public entry points.

Kinds of case (`"kind"`):

  decode   one token per sequence through a stack of layers on resident ring buffers (`NHARingCache.decode`)
  window   one token per sequence with the caller's own window and rotary tables (`fused_recurrent_nha_decode`)
  prompt   inference prefill of a hybrid model's NHA layer (`fused_chunk_nha_prefill`), final state kept for decoding
  chunk    `chunk_nha` without gradients: fixed-length or packed sequences, initial and final states, bf16 or fp32
  train    `chunk_nha` forward and backward
  layer    forward and backward of a `NativeHybridAttention` layer, parameter gradients included
  block    prompt of a hybrid decoder's attention block on a fresh cache (projections, glue, operator, hand-over)

Head shapes are those of the 340M layer (4 heads of 256), the Llama-3-8B-style block (32 / 8 heads of 128), the
Qwen3-MoE-style block (32 / 4 heads of 128) and generic ones; 64 slots throughout.
"""
import torch
import torch.nn.functional as F

import nha_amd
from nha_amd.hybrid import HybridNHAConfig, LlamaNativeHybridAttention, Qwen3MoeNativeHybridAttention
from nha_amd.layer import NativeHybridAttention

M = 64            # slots
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # one user, one token through a stack of four NHA layers of a hybrid model: launches and latency
        dict(name="decode_one", kind="decode", B=1, HQ=32, H=4, D=128, W=64, layers=4),
        # a few users with long windows, not a power of two of them, prompts of different lengths
        dict(name="decode_few", kind="decode", B=3, HQ=32, H=8, D=128, W=2048, layers=1),
        # the serving batch: 128 users, ring buffers full, every ring at its own position
        dict(name="decode_batch", kind="decode", B=128, HQ=32, H=8, D=128, W=1024, layers=1),
        # the stateless decode op as a hybrid model's attention calls it: raw window, tables of each sequence
        dict(name="decode_rotary", kind="window", B=16, HQ=32, H=4, D=128, W=64),
        # a chat prompt of an odd length through one attention block of the MoE-style decoder
        dict(name="block_prompt", kind="block", B=1, T=331, HQ=32, H=4, D=128, W=64, hidden=2048, flavour="qwen"),
        # long prompts through a hybrid model's NHA layer
        dict(name="prompt_hybrid", kind="prompt", B=2, T=8192, HQ=32, H=8, D=128, W=64, dtype="bf16"),
        # long-context prefill with a long window: the largest call
        dict(name="chunk_long", kind="chunk", B=2, T=16384, HQ=32, H=8, D=128, W=2048, shifted=True, packed=False,
             states=False, normalizer=1.0, gate_mean=-1.0, dtype="bf16"),
        # packed documents of 64 to 4096 tokens at the 340M layer's heads, continued from initial states
        dict(name="chunk_packed", kind="chunk", B=1, T=32768, HQ=4, H=4, D=256, W=512, shifted=False, packed=True,
             states=True, normalizer=1.0, gate_mean=0.0, dtype="bf16"),
        # fp32: what a numerics check or an fp32 model runs
        dict(name="chunk_fp32", kind="chunk", B=1, T=512, HQ=4, H=4, D=64, W=64, shifted=True, packed=False, states=True,
             normalizer=1.0, gate_mean=0.0, dtype="fp32"),
        # a training step of the 340M model's layer
        dict(name="layer_340m", kind="layer", B=8, T=2048, hidden=1024, HQ=4, H=4, W=512, packed=False),
        # the operator's training step at the long-context heads
        dict(name="train_long", kind="train", B=2, T=8192, HQ=32, H=8, D=128, W=2048, shifted=True, packed=False,
             normalizer=1.0, gate_mean=-1.0),
        # the operator's training step on a small packed batch of ragged documents, one key head per query head
        dict(name="train_packed", kind="train", B=1, T=5003, HQ=16, H=16, D=64, W=128, shifted=False, packed=True,
             normalizer=8.0, gate_mean=0.0),
    ]


def _log_int(rng, lo, hi):
    """Whole number between lo and hi, uniform in its logarithm."""
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


HEADS = [(32, 8, 128), (32, 4, 128), (8, 2, 128), (16, 16, 128), (8, 4, 128), (4, 4, 256), (8, 2, 256), (16, 16, 64), (16, 4, 64)]
GATES = [(1.0, 0.0), (1.0, -1.0), (8.0, 0.0)]     # normalizer, mean of the gate logits


def draw(rng):
    kind = rng.choice(["decode", "decode", "window", "prompt", "chunk", "chunk", "train", "train", "layer", "block"])
    HQ, H, D = rng.choice(HEADS)
    norm, mean = rng.choice(GATES)
    if kind == "decode":
        return dict(kind=kind, B=_log_int(rng, 1, 128), HQ=HQ, H=H, D=D, W=_log_int(rng, 16, 2048) if D * H <= 512 else
                    _log_int(rng, 16, 1024), layers=rng.choice([1, 1, 4]))
    if kind == "window":
        HQ, H, D = rng.choice([h for h in HEADS if h[2] <= 128])
        return dict(kind=kind, B=_log_int(rng, 1, 64), HQ=HQ, H=H, D=D, W=_log_int(rng, 16, 1024))
    if kind == "prompt":
        if rng.random() < 0.2:
            HQ, H, D = rng.choice([(4, 4, 64), (8, 2, 128), (16, 4, 64)])
            return dict(kind=kind, B=_log_int(rng, 1, 4), T=_log_int(rng, 65, 1024), HQ=HQ, H=H, D=D, W=_log_int(rng, 16, 64),
                        dtype="fp32")
        return dict(kind=kind, B=_log_int(rng, 1, 4), T=_log_int(rng, 65, 8192), HQ=HQ, H=H, D=D, W=_log_int(rng, 16, 64),
                    dtype="bf16")
    if kind == "chunk":
        if rng.random() < 0.25:
            HQ, H, D = rng.choice([(4, 4, 64), (8, 2, 128), (16, 4, 64), (4, 4, 256)])
            return dict(kind=kind, B=1, T=_log_int(rng, 130, 2048), HQ=HQ, H=H, D=D, W=_log_int(rng, 32, 128),
                        shifted=rng.random() < 0.5, packed=rng.random() < 0.5, states=True, normalizer=norm, gate_mean=mean,
                        dtype="fp32")
        packed = rng.random() < 0.5
        return dict(kind=kind, B=1 if packed else _log_int(rng, 1, 4), T=_log_int(rng, 300, 8192), HQ=HQ, H=H, D=D,
                    W=_log_int(rng, 64, 2048), shifted=rng.random() < 0.5, packed=packed, states=rng.random() < 0.5,
                    normalizer=norm, gate_mean=mean, dtype="bf16")
    if kind == "train":
        packed = rng.random() < 0.5
        return dict(kind=kind, B=1 if packed else _log_int(rng, 1, 2), T=_log_int(rng, 500, 6000), HQ=HQ, H=H, D=D,
                    W=_log_int(rng, 64, 1024), shifted=False, packed=packed, normalizer=norm, gate_mean=mean)
    if kind == "layer":
        return dict(kind=kind, B=_log_int(rng, 1, 8), T=_log_int(rng, 200, 2048), W=_log_int(rng, 64, 1024), packed=rng.random() < 0.3,
                    **rng.choice([dict(hidden=1024, HQ=4, H=4), dict(hidden=1024, HQ=8, H=8), dict(hidden=1024, HQ=8, H=2)]))
    flavour = rng.choice(["qwen", "llama"])
    return dict(kind=kind, B=_log_int(rng, 1, 4), T=_log_int(rng, 65, 4096), HQ=32, H=4 if flavour == "qwen" else 8, D=128,
                W=rng.choice([16, 32, 64, 2048]), hidden=2048 if flavour == "qwen" else 4096, flavour=flavour)


# ---- inputs ------------------------------------------------------------------------------------------

class _Draws:
    """Inputs made on the GPU from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV).manual_seed(seed)
        self.host = torch.Generator().manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        return (torch.randn(*shape, generator=self.gen, device=DEV, dtype=torch.float32) * std).to(dtype)

    def gates(self, *shape, normalizer, mean, dtype):
        """Log forget gates and write strengths as the layers form them."""
        g = (F.logsigmoid(self.normal(*shape, dtype=torch.float32) + mean) / normalizer).to(dtype)
        return g, (1 - g.float().exp()).to(dtype)

    def lengths(self, total, lo, hi):
        """As many lengths as `total` holds on average, each between lo and hi, whose sum is `total`."""
        n = max(1, round(2 * total / (lo + hi)))
        while True:
            out = torch.randint(lo, hi + 1, (n - 1,), generator=self.host).tolist()
            last = total - sum(out)
            if n == 1 or lo <= last <= hi:
                return [*out, last]


def _document_lengths(total):
    """Shortest and longest document of a packed batch of `total` tokens."""
    return (64, 4096) if total >= 16384 else (17, max(64, total // 3))


def _boundaries(lens):
    return torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=DEV)


def _operands(case, r, dtype, normalizer, mean):
    """The seven operands of the prefill: the window's rotated q and k, the slots' q and k, v, s, g."""
    B, T, HQ, H, D = (case[k] for k in ("B", "T", "HQ", "H", "D"))
    std = D ** -0.5
    q_swa, q_gsa = (r.normal(B, T, HQ, D, std=std, dtype=dtype) for _ in range(2))
    k_swa, k_gsa, v = (r.normal(B, T, H, D, std=std, dtype=dtype) for _ in range(3))
    g, s = r.gates(B, T, H, M, normalizer=normalizer, mean=mean, dtype=dtype)
    return q_swa, k_swa, q_gsa, k_gsa, v, s, g


def _reset(module, r):
    """Weights of the module from the case's seed (the scale of the default initialisation; norms near one)."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if p.dim() == 1:
                p.copy_(1 + r.normal(*p.shape, std=0.05, dtype=torch.float32))
            else:
                p.copy_(r.normal(*p.shape, std=p.shape[-1] ** -0.5, dtype=torch.float32))


def _prepare_decode(case, r):
    B, HQ, H, D, W = (case[k] for k in ("B", "HQ", "H", "D", "W"))
    cache, steps = nha_amd.NHARingCache(W), []
    lens = torch.randint(W, W + max(2, W // 4), (B,), generator=r.host).tolist()     # prompts that filled their windows
    total, cu = sum(lens), _boundaries(lens)
    for layer in range(case["layers"]):
        k, kg, v = (r.normal(1, total, H, D) for _ in range(3))
        g, _ = r.gates(1, total, H, M, normalizer=8.0, mean=0.0, dtype=torch.bfloat16)
        state = (r.normal(B, H, D, M, std=0.1, dtype=torch.float32), r.normal(B, H, M, D, std=0.1, dtype=torch.float32))
        cache.prefill(layer, k, kg, v, g, state, cu_seqlens=cu)
        q, sq = r.normal(B, HQ, D), r.normal(B, HQ, D)
        k1, kg1, v1 = (r.normal(B, H, D) for _ in range(3))
        g1, _ = r.gates(B, H, M, normalizer=8.0, mean=0.0, dtype=torch.bfloat16)
        steps.append((q, sq, k1, kg1, v1, g1))
    return dict(cache=cache, steps=steps)


def _run_decode(s):
    cache, outs = s["cache"], []
    for layer, args in enumerate(s["steps"]):
        o = cache.decode(layer, *args)
        st = cache.states[layer]
        outs.append((o, st.hk, st.hv, st.ring_k, st.ring_kg, st.ring_v, st.ring_g, st.count))
    return outs


def _prepare_window(case, r):
    B, HQ, H, D, W = (case[k] for k in ("B", "HQ", "H", "D", "W"))
    ends = torch.randint(W, 8 * W, (B,), generator=r.host).to(DEV)
    pos = ends[:, None] - W + 1 + torch.arange(W, device=DEV)[None]
    ang = pos[..., None].float() * (10000.0 ** (-torch.arange(0, D, 2, device=DEV).float() / D))
    ang = torch.cat([ang, ang], -1)
    g, w = r.gates(B, 1, H, M, normalizer=8.0, mean=0.0, dtype=torch.bfloat16)
    return dict(q=r.normal(B, 1, HQ, D), k=r.normal(B, 1, H, D), v=r.normal(B, 1, H, D), g=g, s=w, sw_k=r.normal(B, W, H, D),
                sw_v=r.normal(B, W, H, D), cos=ang.cos().bfloat16(), sin=ang.sin().bfloat16(),
                initial_state=(r.normal(B, H, D, M, std=0.1, dtype=torch.float32),
                               r.normal(B, H, M, D, std=0.1, dtype=torch.float32)))


def _run_window(s):
    return nha_amd.fused_recurrent_nha_decode(**s, output_final_state=True)


def _prepare_prompt(case, r):
    q_swa, k_swa, q, k, v, s, g = _operands(case, r, DTYPES[case["dtype"]], 8.0, 0.0)
    return dict(q=q, k=k, v=v, rotary_q=q_swa, rotary_k=k_swa, s=s, g=g, window_size=case["W"])


def _run_prompt(s):
    return nha_amd.fused_chunk_nha_prefill(**s, output_final_state=True)


def _prepare_chunk(case, r):
    dtype = DTYPES[case.get("dtype", "bf16")]
    ops = _operands(case, r, dtype, case["normalizer"], case["gate_mean"])
    kw = dict(window_size_left=case["W"] - 1, gsa_kv_shift=case["W"]) if case["shifted"] else dict(window_size_left=case["W"])
    n = case["B"]
    if case["packed"]:
        lens = r.lengths(case["T"], *_document_lengths(case["T"]))
        kw["cu_seqlens"] = _boundaries(lens)
        n = len(lens)
    if case.get("states"):
        kw["initial_state"] = (r.normal(n, case["H"], case["D"], M, std=0.1, dtype=torch.float32),
                               r.normal(n, case["H"], M, case["D"], std=0.1, dtype=torch.float32))
        kw["output_final_state"] = True
    return ops, kw


def _run_chunk(s):
    ops, kw = s
    return nha_amd.chunk_nha(*ops, **kw)


def _prepare_train(case, r):
    ops, kw = _prepare_chunk(case, r)
    do = r.normal(case["B"], case["T"], case["HQ"], case["D"])
    return [x.requires_grad_() for x in ops], kw, do


def _run_train(s):
    ops, kw, do = s
    o = nha_amd.chunk_nha(*ops, **kw)[0]
    return o.detach(), torch.autograd.grad(o, ops, do)


def _prepare_layer(case, r):
    layer = NativeHybridAttention(hidden_size=case["hidden"], num_heads=case["HQ"], num_kv_heads=case["H"], num_slots=M,
                                  layer_idx=0, window_size=case["W"]).to(DEV)
    _reset(layer, r)
    layer = layer.to(torch.bfloat16).train()
    B, T = case["B"], case["T"]
    kw = {}
    if case["packed"]:
        kw["cu_seqlens"] = _boundaries(r.lengths(B * T, *_document_lengths(B * T)))
        B, T = 1, B * T
    x = r.normal(B, T, case["hidden"], std=0.5).requires_grad_()
    return layer, x, r.normal(B, T, case["hidden"]), kw


def _run_layer(s):
    layer, x, dy, kw = s
    y = layer(x, **kw)[0]
    return y.detach(), torch.autograd.grad(y, [x, *layer.parameters()], dy)


def _prepare_block(case, r):
    full = case["W"] > 64
    cfg = HybridNHAConfig(hidden_size=case["hidden"], num_attention_heads=case["HQ"], num_key_value_heads=case["H"],
                          head_dim=case["D"], num_slots=M, window_size=64 if full else case["W"],
                          block_size=1 if full else None, transformer_idx=0 if full else None)
    block = (Qwen3MoeNativeHybridAttention if case["flavour"] == "qwen" else LlamaNativeHybridAttention)(cfg, 0).to(DEV)
    _reset(block, r)
    block = block.to(torch.bfloat16).eval()
    x = r.normal(case["B"], case["T"], case["hidden"], std=0.5)
    pos = torch.arange(case["T"], device=DEV)[None].expand(case["B"], -1)
    return block, x, pos


@torch.no_grad()
def _run_block(s):
    block, x, pos = s
    cache = nha_amd.NHACache()
    y = block(x, position_ids=pos, past_key_value=cache, use_cache=True)[0]
    st = cache.states[0]
    return y, st.hk, st.hv, st.ring_k, st.ring_kg, st.ring_v, st.ring_g, st.count


_PREPARE = dict(decode=_prepare_decode, window=_prepare_window, prompt=_prepare_prompt, chunk=_prepare_chunk,
                train=_prepare_train, layer=_prepare_layer, block=_prepare_block)
_RUN = dict(decode=_run_decode, window=_run_window, prompt=_run_prompt, chunk=_run_chunk, train=_run_train, layer=_run_layer,
            block=_run_block)


def prepare(case, seed):
    return case["kind"], _PREPARE[case["kind"]](case, _Draws(seed))


def run(state):
    kind, s = state
    return _RUN[kind](s)


# ---- what a pass cannot do without -------------------------------------------------------------------

def _prefill_work(B, T, HQ, H, D, W, size=2, states=0, lse=False, window_only=False):
    tokens = B * T
    w = sum(min(t + 1, W) for t in range(T)) / T
    reads = tokens * (2 * HQ * D + 3 * H * D + 2 * H * M) * size
    writes = tokens * HQ * D * size + (8 * tokens * HQ if lse else 0)
    flops = tokens * HQ * (8 * D * M + 4 * w * D) + 4 * tokens * H * D * M
    if window_only:
        flops = tokens * HQ * 4 * w * D
    return dict(bytes=reads + writes + 8 * B * H * D * M * states, flops=flops)


def work(case):
    kind, H, HQ = case["kind"], case["H"], case["HQ"]
    if kind in ("decode", "window"):
        B, D, W, n = case["B"], case["D"], case["W"], case.get("layers", 1)
        state = 2 * 8 * B * H * D * M
        window = 4 * B * W * H * D
        small = 2 * B * (3 * HQ * D + 2 * H * (3 * D + M))
        tables = 4 * B * W * D if kind == "window" else 0
        return dict(bytes=n * (state + window + small + tables), flops=n * B * (HQ * (4 * D * M + 4 * W * D) + 8 * H * D * M))
    if kind == "prompt":
        return _prefill_work(case["B"], case["T"], HQ, H, case["D"], case["W"], 4 if case["dtype"] == "fp32" else 2, states=1)
    if kind in ("chunk", "train"):
        # packed sequences: the lengths differ from seed to seed; their mean stands for them
        B, T = case["B"], case["T"]
        length = max(1, sum(_document_lengths(T)) // 2) if case["packed"] else T
        w = _prefill_work(B * T / length, length, HQ, H, case["D"], case["W"], 4 if case.get("dtype") == "fp32" else 2,
                          states=2 if case.get("states") else 0, lse=kind == "chunk")
        if kind == "train":
            # backward: the forward's products twice and once more (scores recomputed); operands, output and its gradient
            # read, the gradients of the operands written
            tokens = B * T
            return dict(bytes=w["bytes"] + 2 * tokens * (2 * (2 * HQ * case["D"] + 3 * H * case["D"] + 2 * H * M) + 2 * HQ * case["D"]),
                        flops=3.5 * w["flops"])
        return w
    hidden = case["hidden"]
    tokens = case["B"] * case["T"]
    if kind == "layer":
        D = hidden // HQ
        ext = hidden * (HQ * D + 2 * H * D + H * M + HQ * D)          # projection weights
        length = sum(_document_lengths(tokens)) // 2 if case["packed"] else case["T"]
        w = _prefill_work(tokens / length, length, HQ, H, D, case["W"])
        return dict(bytes=2 * (4 * tokens * hidden + 2 * ext), flops=6 * tokens * ext + 3.5 * w["flops"])
    D, full = case["D"], case["W"] > 64
    ext = hidden * (2 * HQ * D + 2 * H * D + (0 if full else H * M))
    w = _prefill_work(case["B"], case["T"], HQ, H, D, case["W"], window_only=full)
    ring = 2 * case["B"] * case["W"] * H * (3 * D + M) + 8 * case["B"] * H * D * M
    return dict(bytes=2 * (2 * tokens * hidden + ext) + ring, flops=2 * tokens * ext + w["flops"])


def tolerance(case):
    """About four times what the bf16 paths were seen to differ from the same path in fp32 on the same inputs, over the
    listed cases and 40 drawn ones (relative 2-norm, largest difference; worst output of each): decode 2.2e-3 / 8e-3,
    window 3.2e-3 / 1.5e-2, prefill 2.5e-3 / 3.3e-2, gradients of the operator 1.0e-2 / 0.15 (the gates' gradients are
    differences of large sums), layer 1.4e-2 / 0.12 and block 1.3e-2 / 0.07 (their projections' roundings included).  fp32
    against the oracle at T = 512: 7e-7 / 5e-6, sums over longer ranges and exponentials of larger arguments allowed for."""
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"decode": {"rel": 0.009, "max": 0.035}, "window": {"rel": 0.013, "max": 0.06}, "prompt": {"rel": 0.01, "max": 0.13},
            "chunk": {"rel": 0.01, "max": 0.13}, "train": {"rel": 0.03, "max": 0.6}, "layer": {"rel": 0.03, "max": 0.5},
            "block": {"rel": 0.03, "max": 0.3}}[case["kind"]]
