// Window branch of the NHA prefill backward for K == V == D == 128 (bf16) with four (or a multiple of
// four) query heads per kv-head: the data movement of ring_out_kernel (prefill_ring.hip) applied to the
// products of bwd_dq_kernel / bwd_dkv_kernel (prefill_bwd_mfma.hip; the part
// nha_fla/ops/nha/chunk.py:499-511 hands to flash-attn's backward).  With the merged log-sum-exp and
// delta = do . o of the whole op per (token, q-head), window logits w = scale q.k:
//   pi = e^(w - lse),  dw = pi (do.v - delta),
//   dq_swa_q = scale sum_j dw k_j,   dk_swa_j = scale sum_q dw q_q,   dv_j += sum_q pi do_q.
// Every streamed operand goes from global memory straight into LDS (global_load_lds_dwordx4) through a ring of buffers.  One
// layout of a tile serves row fragments and transposing reads: 1 KB blocks of 16 rows x 32 columns, of 64-byte rows with their
// pieces exchanged (LineTile) in ring_dq_kernel, two planes of 32-byte rows in ring_dkv_kernel (with LineTile 905 -> 920 us).
//
// ring_dq_kernel: one workgroup of 8 waves = one 64-token chunk x 4 query heads of one kv-head (a query
//   per lane, 32 queries per wave), so the K / V rows of the window are fetched once for the four heads,
//   in units of 32 keys: a K tile (row fragments for S^T = K Q^T, transposed for dQ^T += K^T dS^T) and a V tile (row
//   fragments for dP^T = V dO^T).  Two units share a barrier, and the products of the two interleave with what
//   lies between them: exponentials beside dP, dS of the first unit beside the scores of the second, dS of the second
//   beside dQ of the first.  It also
//   leaves (-lse / scale, -delta) per (token, q-head) as pairs for the kernel below, whose score and
//   dP accumulators start from them.
//   Bound: as below, 56 % of the matrix rate.  B=2, T=8192, 32/8 heads, W=2048: 625 us unit by unit with K in LDS twice and
//   the compiler's schedule, 597 like this, 591 with a stretch's first fragments requested during the stretch before, 575 (582 on that card) with the
//   query and do rows loaded in whole lines: 2 x 4096 tokens, W=256 114 -> 110, 500 tokens 25.7 -> 23.7, 1700 tokens, W=64 19.5 -> 19.8.
// ring_dkv_kernel: one workgroup of 8 waves = 256 keys of one kv-head (a key per lane and 16-key block, 32 keys per wave, K
//   rows in registers, V rows in LDS); the q / do rows of every query head of the group stream through the ring in items of
//   32 queries: a tile of each plus the 32 (lse, delta) pairs.  One layout of a tile serves both reads, the row fragments of
//   S = Q K^T and dP = dO V^T and the transposing read of dV^T += dO^T P and dK^T += Q^T dS.
//   The first and the last units of a head are triangles over the waves (causal edge, window edge) that
//   complement each other: such units are held in LDS two at a time and every wave works on its own.
//   Bound: the products and, beside them, LDS reads and exponentials of two waves per SIMD (48 % of the matrix rate over the
//   launch).  B=2, T=8192, 32/8 heads, W=2048: 1149 us with K and V in registers (no room to read ahead; the row
//   fragments read once per 16-key block), each tile in LDS twice and the exponentials between the products; 950 with
//   V in LDS, one tile and one stream of products; 934 with two items per barrier.  Transposed fragments one, three or four
//   products ahead instead of two: the same.
#include "common.h"
#include "mfma_common.h"

#include <mutex>

namespace nha {
namespace {
using namespace mf;

struct DqP {
  const bf16_t *q, *k, *v, *dout;          // q_swa [T,HQ,D]; k_swa, v [T,H,D]; dout [T,HQ,D]
  const float *lse_swa, *lse_gsa, *delta;  // [T,HQ]
  float2* ld;                              // [T,HQ] out: (-lse / scale, -delta) of the merged softmax
  bf16_t* dq;
  const int32_t *cu, *cidx;
  int HQ, H, NG, NT, wl;
  float scale;
};

constexpr int D = 128;
constexpr int KS = D / 32;            // contraction steps of the score products
constexpr int DB = D / 16;            // 16-row blocks of dQ^T
constexpr int UB = 32 * D * 2;        // bytes of a 32-row tile
constexpr int HB = UB / 2;
constexpr int NR = 4;                 // ring slots of ring_dkv_kernel
constexpr int NRU = 8;                // ring slots of ring_dq_kernel
constexpr int UNIT = 2 * UB;          // K tile | V tile
constexpr int LPW = 2;                // LDS-direct loads per wave and unit (16 blocks of 1 KB, 8 waves)
constexpr int BYTES = NRU * UNIT;
constexpr int RQB = 2;                // 16-row query blocks per wave

// RAW: the forward of the call formed its scores from queries that were not scaled, and rounded, before the products (ring_out_kernel with
// one 16-row block per wave), and so do these: with rounded ones dq of calls of strong logits was up to a sixth further from 64 bits.
template <bool RAW>
__global__ __launch_bounds__(512, 1) void ring_dq_kernel(const DqP p) {
  extern __shared__ __align__(1024) unsigned char smem_[];
  lbyte* const lds = (lbyte*)smem_;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kb = lane >> 4;
  const int H = p.H, HQ = p.HQ, NG = p.NG;
  // grid = (kv-head x group of four q-heads, chunk), chunks from the last to the first
  const int ngrp = NG / 4;
  int vx, vy;
  xcd_tile(ngrp, p.NT, vx, vy);
  const int chunk = p.NT - 1 - vy;
  const int h = vx / ngrp, grp = vx % ngrp;
  const int hq = h * NG + grp * 4 + wave / 2;
  const int qb0 = (wave % 2) * RQB;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int c0 = bos + it * BT;
  const int rows = (eos - c0) < BT ? (eos - c0) : BT;
  const float cs = p.scale * LOG2E;

  // unit u covers keys [c0 + 32 - 32 u, c0 + 64 - 32 u); c0 - bos is a multiple of 64, so no unit starts
  // before its sequence; units 0 and 1 are the chunk's own rows and may run past eos
  int lowest = bos;
  if (p.wl >= 0 && c0 - p.wl > bos) lowest = c0 - p.wl;
  // an even number: the loop takes them in twos, and (c0 - bos) / 32 is even, so the one added does not start before its
  // sequence either (the window masks it)
  const int nunits = ((c0 + 64 - lowest + 31) / 32 + 1) & ~1;

  // a unit's blocks of 16 rows x 32 columns, one of each tile per wave: half wave / KS, columns 32 (wave % KS) ..
  const int rh = wave / KS, cq = wave % KS;
  const bf16_t* const kbase = p.k + ((int64_t)bos * H + h) * D;
  const bf16_t* const vbase = p.v + ((int64_t)bos * H + h) * D;
  const uint32_t pcol = LineTile<D>::load_col(cq, lane);
  // rows past eos (units 0 and 1 only) are read from row eos - 1: always masked, always finite
  auto issue_unit = [&](int u) {
    int row = c0 + 32 - 32 * u + 16 * rh + LineTile<D>::load_row(lane);
    row = row < eos ? row : eos - 1;
    const uint32_t off = ((uint32_t)(row - bos) * (uint32_t)(H * D) + pcol) * 2;
    const uint32_t dst = lds0 + (u & (NRU - 1)) * UNIT + rh * HB + cq * 1024;
    g2l16(kbase, off, dst);
    g2l16(vbase, off, dst + UB);
  };
#pragma unroll
  for (int u = 0; u < NRU - 2; ++u)
    if (u < nunits) issue_unit(u);

  // query-side fragments: q pre-scaled by scale * log2(e) unless RAW (the rounding the forward's scores saw), do as it is.  The rows come in
  // whole lines, as 1 KB blocks of 16 rows x 32 columns (a fragment as it lies in memory, 16 bytes of 16 rows, takes three
  // times as long to load), and are put into fragment order through the two ring slots that no unit has been requested into.
  uint4 qraw[RQB][KS], draw[RQB][KS];
#pragma unroll
  for (int qb = 0; qb < RQB; ++qb) {
    int r = 16 * (qb0 + qb) + LineTile<D>::load_row(lane);
    r = r < rows ? r : rows - 1;
    const int64_t at = ((int64_t)(c0 + r) * HQ + hq) * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qraw[qb][ks] = *reinterpret_cast<const uint4*>(p.q + at + LineTile<D>::load_col(ks, lane));
      draw[qb][ks] = *reinterpret_cast<const uint4*>(p.dout + at + LineTile<D>::load_col(ks, lane));
    }
  }
  const uint32_t own = (NRU - 2) * UNIT + wave * 4096, kaddr = LineTile<D>::row_at(lane);
  auto turned = [&](const uint4& x, int slot) {   // (what a wave writes there it alone reads)
    *reinterpret_cast<NHA_LDS u32x4*>(lds + (own + slot * 1024 + lane * 16)) = __builtin_bit_cast(u32x4, x);
    return *reinterpret_cast<const NHA_LDS u32x4*>(lds + (own + slot * 1024 + kaddr));
  };
  bf16x8 qf[RQB][KS], df[RQB][KS];
  float nlse[RQB], dl[RQB];
#pragma unroll
  for (int qb = 0; qb < RQB; ++qb) {
    const int irow = 16 * (qb0 + qb) + l16;
    const bool valid = irow < rows;
    const int64_t tq = (int64_t)(c0 + (valid ? irow : 0)) * HQ + hq;
    const uint32_t on = valid ? ~0u : 0u;   // (a mask: a choice between loaded registers may become a branch)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 x = turned(qraw[qb][ks], (2 * ks) & 3) & on;
      bf16x8 r;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = __uint_as_float((e & 1) ? (x[e >> 1] & 0xffff0000u) : (x[e >> 1] << 16));
        r[e] = (__bf16)(f * cs);
      }
      qf[qb][ks] = RAW ? __builtin_bit_cast(bf16x8, x) : r;
      df[qb][ks] = __builtin_bit_cast(bf16x8, turned(draw[qb][ks], (2 * ks + 1) & 3) & on);
    }
    float ls = 0.f, lg = 0.f;
    if (valid) {
      ls = p.lse_swa[tq];
      lg = p.lse_gsa[tq];
    }
    const float mx = fmaxf(ls, lg);
    nlse[qb] = valid ? -(mx + __logf(__expf(ls - mx) + __expf(lg - mx))) * LOG2E : 0.f;
    dl[qb] = valid ? p.delta[tq] : 0.f;
    if (valid && kb == 0) p.ld[tq] = make_float2(nlse[qb] / cs, -dl[qb]);
  }
  f32x4 dQ[DB][RQB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int qb = 0; qb < RQB; ++qb) dQ[db][qb] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const uint32_t vaddr = LineTile<D>::col_at(lane);
  // row fragment of a tile at byte address a: rows 16 kk + l16, columns 32 ks + 8 kb ..
  auto rfrag = [&](uint32_t a, int kk, int ks) -> bf16x8 {
    return *reinterpret_cast<const NHA_LDS bf16x8*>(lds + (a + kaddr) + kk * HB + ks * 1024);
  };
  // transposed fragment: X[4 kb + e][16 db + l16] (e < 4) and X[16 + 4 kb + e - 4][..]
  auto tfrag = [&](uint32_t a, int db) -> bf16x8 {
    const lbyte* pa = lds + ((a + vaddr) ^ ((db & 1) * 32)) + (db >> 1) * 1024;
    struct { s16x4 a, b; } t;
    t.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pa);
    t.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)(pa + HB));
    return __builtin_bit_cast(bf16x8, t);
  };
  auto is_edge = [&](int u) -> bool { return (63 - 32 * u > 0) || (p.wl >= 0 && 32 - 32 * u < 63 - p.wl); };

  // The products of a unit as stretches that other work runs beside; scores (16-key block kk, 16-query block qb) at 2 kk + qb.
  // A stretch is given its first fragments, and its last product is preceded by `tail`, the request for the next stretch's.
  constexpr int NQ = 2 * RQB;
  struct Unit {
    f32x4 S[NQ], dP[NQ];
    bf16x8 dS[RQB];
  };
  struct Frags {
    bf16x8 x[2];
  };
  constexpr int PT = 2;   // transposed fragments are requested this many products ahead
  auto row_frags = [&](uint32_t a, int ks) { return Frags{{rfrag(a, 0, ks), rfrag(a, 1, ks)}}; };
  auto columns = [&](uint32_t a) { return Frags{{tfrag(a, 0), tfrag(a, 1)}}; };
  auto scores = [&](Unit& t, uint32_t base, const Frags& first, auto beside, auto tail) {   // S = K Q^T - lse
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const float from = RAW ? 0.f : nlse[q & 1];
      t.S[q] = (f32x4){from, from, from, from};
    }
    Frags ka[KS];
    ka[0] = first;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      __builtin_amdgcn_sched_barrier(0);
      if (ks + 1 < KS) ka[ks + 1] = row_frags(base, ks + 1);
      else tail();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < NQ; ++q) t.S[q] = mfma16(ka[ks].x[q >> 1], qf[q & 1][ks], t.S[q]);
      beside(ks);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mask = [&](Unit& t, int u) {
    if constexpr (RAW)
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) t.S[q][r] = t.S[q][r] * cs + nlse[q & 1];
    if (!is_edge(u)) return;
    const int xbase = 32 - 32 * u;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int y = 16 * (qb0 + (q & 1)) + l16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = xbase + 16 * (q >> 1) + 4 * kb + r;
        const bool ok = (x <= y) && (p.wl < 0 || x >= y - p.wl);
        if (!ok) t.S[q][r] = -INFINITY;
      }
    }
  };
  auto dprob = [&](Unit& t, uint32_t base, const Frags& first, auto tail) {   // dP = V dO^T - delta, the exponentials beside it
#pragma unroll
    for (int q = 0; q < NQ; ++q) t.dP[q] = (f32x4){-dl[q & 1], -dl[q & 1], -dl[q & 1], -dl[q & 1]};
    Frags va[KS];
    va[0] = first;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      __builtin_amdgcn_sched_barrier(0);
      if (ks + 1 < KS) va[ks + 1] = row_frags(base + UB, ks + 1);
      else tail();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < NQ; ++q) t.dP[q] = mfma16(va[ks].x[q >> 1], df[q & 1][ks], t.dP[q]);
#pragma unroll
      for (int r = 0; r < 4; ++r) t.S[ks][r] = fexp2(t.S[ks][r]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto form_ds = [&](Unit& t, int qb) {
    t.dS[qb] = pack8(t.S[qb] * t.dP[qb], t.S[2 + qb] * t.dP[2 + qb]);
  };
  auto dquery = [&](Unit& t, uint32_t base, const Frags& first, auto beside, auto tail) {   // dQ^T[d][q] += K^T[d][key] dS^T[key][q]
    bf16x8 kt[DB] = {first.x[0], first.x[1]};
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      __builtin_amdgcn_sched_barrier(0);
      if (db + PT < DB) kt[db + PT] = tfrag(base, db + PT);
      else if (db + 1 == DB) tail();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int qb = 0; qb < RQB; ++qb) dQ[db][qb] = mfma16(kt[db], t.dS[qb], dQ[db][qb]);
      beside(db);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  for (int u = 0; u < nunits; u += 2) {
    // units u and u + 1 have landed (this wave's part), then everybody's; the four after them may stay in flight
    if (u + 4 < nunits) wait_vm<4 * LPW>();
    else if (u + 2 < nunits) wait_vm<2 * LPW>();
    else wait_vm<0>();
    lds_barrier();
    // every wave is past units u - 1 and u - 2: their slots take the next two
    if (u + NRU - 2 < nunits) {
      issue_unit(u + NRU - 2);
      issue_unit(u + NRU - 1);
    }
    const uint32_t b0 = (uint32_t)((u & (NRU - 1)) * UNIT), b1 = b0 + UNIT;   // (u is even, so is NRU)
    Unit t0, t1;
    Frags k0 = row_frags(b0, 0), v0, k1, v1, c0f, c1f;
    scores(t0, b0, k0, [](int) {}, [&] { v0 = row_frags(b0 + UB, 0); });
    mask(t0, u);
    dprob(t0, b0, v0, [&] { k1 = row_frags(b1, 0); });
    scores(t1, b1, k1, [&](int ks) { if (ks >= 1 && ks <= RQB) form_ds(t0, ks - 1); }, [&] { v1 = row_frags(b1 + UB, 0); });
    mask(t1, u + 1);
    dprob(t1, b1, v1, [&] { c0f = columns(b0); });
    dquery(t0, b0, c0f, [&](int db) { if (db >= 1 && db <= RQB) form_ds(t1, db - 1); }, [&] { c1f = columns(b1); });
    dquery(t1, b1, c1f, [](int) {}, [] {});
  }
#pragma unroll
  for (int qb = 0; qb < RQB; ++qb) {
    const int irow = 16 * (qb0 + qb) + l16;
    if (irow >= rows) continue;
    bf16_t* op = p.dq + ((int64_t)(c0 + irow) * HQ + hq) * D + 4 * kb;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      bf16x4 pk;
#pragma unroll
      for (int r = 0; r < 4; ++r) pk[r] = (__bf16)(dQ[db][qb][r] * p.scale);
      *reinterpret_cast<bf16x4*>(op + 16 * db) = pk;
    }
  }
}

// ------------------------------------------------------------------------------------------------------
struct DkvP {
  const bf16_t *q, *k, *v, *dout;          // q_swa [T,HQ,D]; k_swa, v [T,H,D]; dout [T,HQ,D]
  const float2* ld;                        // [T,HQ] (-lse / scale, -delta): what the two score accumulators start from
  const float* dvs;                        // [T,H,D] slot-branch part of dv
  bf16_t *dk, *dv;
  float *wk, *wv;                          // PARTS: in their place fp32 sums, [gridDim.z][T,H,D] (pd floats each)
  int64_t pd;
  const int32_t *cu, *cidx;
  int HQ, H, NG, NT, wl;                   // NG: query heads of a workgroup (PARTS: a kv-head's are shared out over gridDim.z)
  float scale;
};

// an item: q tile | do tile | 32 (lse, delta) pairs
constexpr int KV_Q = 0, KV_O = UB, KV_LD = 2 * UB, KV_ITEM = 2 * UB + 256;
template <int G> constexpr int KV_NR = G == 2 ? 7 : 4;   // items in LDS
template <int KEYS, int G> constexpr int KV_BYTES = KV_NR<G> * KV_ITEM + KEYS * D * 2;   // ring, then the V rows of the workgroup's keys

// waits until at most `younger` items' requests of this wave are in flight
template <int LPW, int G>
__device__ __forceinline__ void wait_items(int younger) {
  if (G == 2 && younger >= 5) wait_vm<5 * LPW>();
  else if (G == 2 && younger == 4) wait_vm<4 * LPW>();
  else if (G == 2 && younger == 3) wait_vm<3 * LPW>();
  else if (younger >= 2) wait_vm<2 * LPW>();
  else if (younger == 1) wait_vm<LPW>();
  else wait_vm<0>();
}

// KEYS: keys per workgroup, 256 or 128, G: the waves in G groups, each with all keys and every G-th item, whose sums are added at the end.
// A wave with 32 keys feeds two matrix products with every q / do fragment it reads from LDS, one with 16 keys (128, G = 1) only one:
// long windows are bound by those reads (B=2, T=8192, 32/8 heads, W=2048: 256 keys 1.17 ms, 128 1.5, 128 in two groups 1.26).  Windows up
// to 160 keys, where a workgroup's walk is a few items long, take 128 keys and one group (W=64 145 us, two groups 169); two groups are
// for calls whose groups of 256 keys leave CUs without work (key_groups): 4000 tokens, W=1000 263 -> 172 us, 233 with bwd_dkv_kernel.
template <int KEYS, int G, bool PARTS>
__global__ __launch_bounds__(512, 1) void ring_dkv_kernel(const DkvP p) {
  constexpr int KW = 8 / G;                // waves that hold the keys, each of G groups all of them
  constexpr int NKB = KEYS / 16 / KW;      // 16-key blocks per wave
  constexpr int NR = KV_NR<G>;
  constexpr int CPG = KEYS / 64;           // chunks per key group
  constexpr int UPG = KEYS / 32;           // 32-query units that a key group spans
  constexpr int KV_LPW = 2;                // tile loads per wave and item (16 blocks of 1 KB, 8 waves)
  extern __shared__ __align__(1024) unsigned char smem_[];
  lbyte* const lds = (lbyte*)smem_;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kb = lane >> 4;
  const int kw = wave % KW, grp = wave / KW;
  const int H = p.H, HQ = p.HQ, NG = p.NG;
  // grid = (kv-head, chunk): the workgroup of every CPG-th chunk of a sequence (every fourth, at 256 keys) takes that
  // chunk and the next CPG - 1; the others leave at once.  Workgroups are handed to the shader engines in turn, in
  // launch order: were the working ones every fourth of that order they would all land on the same engine.  The
  // launch order therefore walks the chunks with stride CPG (chunks 0, 4, 8, ... first, then 1, 5, 9, ...), so that
  // the chunks of a sequence that start a key group are neighbours in it; chunks from the last to the first.
  const int nq = (p.NT + CPG - 1) / CPG;
  const int cperm = CPG * (blockIdx.y % nq) + blockIdx.y / nq;
  if (cperm >= p.NT) return;
  const int chunk = p.NT - 1 - cperm;
  const int h = blockIdx.x, hq0 = PARTS ? (h * gridDim.z + blockIdx.z) * NG : h * NG;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  if (it & (CPG - 1)) return;
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int c0 = bos + it * BT;
  const int kspan = (eos - c0) < KEYS ? (eos - c0) : KEYS;
  const float cs = p.scale * LOG2E;
  // queries that see a key of the workgroup: [c0, qend), in items of 32 per query head
  int qend = eos;
  if (p.wl >= 0 && c0 + kspan + p.wl < eos) qend = c0 + kspan + p.wl;
  const int nun = (qend - c0 + 31) / 32;   // >= 1
  const int total = NG * nun;

  // block (16-row half wave / 4, 32-column block wave % 4) of both tiles of an item
  const int rh = wave >> 2, cq = wave & 3;
  // item (g, u): rows [c0 + 32 u, c0 + 32 u + 32) of query head hq0 + g; rows past eos are read from row
  // eos - 1 (always masked, always finite)
  auto issue_item = [&](int g, int u, int slot) {
    // what follows from the lane number is derived again at every request: kept across the loop it would
    // cost registers the accumulators need
    int ln = threadIdx.x & 63;
    asm volatile("" : "+v"(ln));
    const int hq = hq0 + g;
    const int q0 = c0 + 32 * u;
    const bf16_t* const qbase = p.q + ((int64_t)bos * HQ + hq) * D;
    const bf16_t* const obase = p.dout + ((int64_t)bos * HQ + hq) * D;
    int rt = q0 + 16 * rh + ((ln & 31) >> 1);
    rt = rt < eos ? rt : eos - 1;
    const uint32_t off = ((uint32_t)(rt - bos) * (uint32_t)(HQ * D) + (uint32_t)(4 * cq + 2 * (ln >> 5) + (ln & 1)) * 8) * 2;
    const uint32_t dst = lds0 + slot * KV_ITEM + rh * HB + cq * 1024;
    g2l16(qbase, off, dst + KV_Q);
    g2l16(obase, off, dst + KV_O);
    if (wave == 0) {
      int r = q0 + (ln >> 1);
      r = r < eos ? r : eos - 1;
      g2l4(p.ld, (uint32_t)(((int64_t)r * HQ + hq) * 2 + (ln & 1)) * 4u, lds0 + slot * KV_ITEM + KV_LD);
    }
  };
  // The workgroups of neighbouring key groups of a sequence run at the same time on one XCD, and their
  // query ranges overlap by all but 8 units.  Each walks the units of a head cyclically, starting where
  // the walk of the sequence's first key group would be at that moment: neighbours then request the same
  // q / do rows at about the same time and the second request finds them in L2.
  const int rot = (nun - (UPG * (it / CPG)) % nun) % nun;
  // Complementary units.  Against the 256 keys of the workgroup the first units of a head are triangles (wave w has
  // work in unit u only if w <= u: the queries of a unit must not all lie before the wave's keys) and so are the last
  // ones (the keys must not all have left the window: unit a + K0 has work only for the waves w >= a + 1), and a
  // workgroup takes as long over a unit as its busiest wave.  Units a < npair are therefore worked on together with
  // unit a + K0: both are in LDS at once and every wave takes the one it has work in, never both.
  const int K0 = p.wl >= 0 ? (p.wl + 63) / 32 : 0;
  int npair = 0;
  if (p.wl >= 0 && K0 >= UPG - 1 && nun > K0) npair = (nun - K0) < UPG - 1 ? (nun - K0) : UPG - 1;
  // the walk of a head: its units in cyclic order from rot, the second units of the pairs left out
  auto walk_skip = [&](int x) {
    if (x >= nun) x -= nun;
    if (x >= K0 && x < K0 + npair) {   // empty range without pairs
      x = K0 + npair;
      if (x >= nun) x -= nun;
    }
    return x;
  };
  const int rot0 = walk_skip(rot);
  struct Walk { int g, u, cnt; };
  auto advance = [&](Walk& w) {
    w.cnt += (w.u < npair) ? 2 : 1;
    w.u = walk_skip(w.u + 1);
    if (w.cnt == nun) {
      w.cnt = 0;
      w.u = rot0;
      ++w.g;
    }
  };
  // requests, in the order the loop below consumes the items: the unit of a step, then the unit paired with it
  Walk pw = {0, rot0, 0};
  int pend_u = -1, pend_g = 0;
  auto issue_next = [&](int slot) {
    if (pend_u >= 0) {
      issue_item(pend_g, pend_u, slot);
      pend_u = -1;
      return;
    }
    issue_item(pw.g, pw.u, slot);
    if (pw.u < npair) {
      pend_u = pw.u + K0;
      pend_g = pw.g;
    }
    advance(pw);
  };
  // This lane's keys (one per 16-key block of the wave) and their K / V rows (B operands: K[key][32 ks + 8 kb ..]).  The V rows
  // lie in LDS, in the order in which their wave reads them; K and V both in registers would leave none to read ahead with.
  const int kbase = 16 * NKB * kw;               // first key of the wave, relative to c0
  const uint32_t vrows = (uint32_t)(NR * KV_ITEM + kw * (NKB * KS * 1024));
#pragma unroll
  for (int k2 = 0; k2 < NKB / G; ++k2) {
    const int kk = G == 1 ? k2 : grp;
    const int tk = c0 + kbase + 16 * kk + l16;
    const uint32_t row = (uint32_t)((tk < eos ? tk : eos - 1) - bos) * (uint32_t)(H * D);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      g2l16(p.v + ((int64_t)bos * H + h) * D, (row + 32 * ks + 8 * kb) * 2, lds0 + vrows + (kk * KS + ks) * 1024);
  }
  int issued = 0, islot = 0, cslot = 0;   // items requested; slots of the next request and of item k below
  for (; issued < NR - 1 && issued < total; ++issued) issue_next(islot++);

  bf16x8 kfr[NKB][KS];
#pragma unroll
  for (int kk = 0; kk < NKB; ++kk) {
    const int tk = c0 + kbase + 16 * kk + l16;
    const int64_t jk = (int64_t)(tk < eos ? tk : eos - 1) * H + h;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kfr[kk][ks] = as_bf16x8(*reinterpret_cast<const uint4*>(p.k + jk * D + 32 * ks + 8 * kb));
  }
  // the K rows are in their registers before the loop starts: left to the compiler, the wait for them sits
  // at their first use inside the loop, as a wait for every load in flight, the LDS-direct ones included
#pragma unroll
  for (int kk = 0; kk < NKB; ++kk)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(kfr[kk][ks]));
  f32x4 dK[DB][NKB], dV[DB][NKB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int kk = 0; kk < NKB; ++kk) {
      dK[db][kk] = (f32x4){0.f, 0.f, 0.f, 0.f};
      dV[db][kk] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
  uint32_t kaddr, vaddr, faddr;   // set per item (see issue_item)
  // row fragment of a tile at byte address a: rows 16 qb + l16, columns 32 ks + 8 kb ..
  auto rfrag = [&](uint32_t a, int qb, int ks) -> bf16x8 {
    return *reinterpret_cast<const NHA_LDS bf16x8*>(lds + (a + kaddr) + qb * HB + ks * 1024);
  };
  auto vfrag = [&](int kk, int ks) -> bf16x8 {
    return *reinterpret_cast<const NHA_LDS bf16x8*>(lds + faddr + (kk * KS + ks) * 1024);
  };
  auto tfrag = [&](uint32_t a, int db) -> bf16x8 {
    const lbyte* pa = lds + (a + vaddr) + (db >> 1) * 1024 + (db & 1) * 512;
    struct { s16x4 a, b; } t;
    t.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pa);
    t.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)(pa + HB));
    return __builtin_bit_cast(bf16x8, t);
  };

  // queries [32 u, 32 u + 32) against keys [kbase, kbase + 16 NKB), both relative to c0: nothing to do if
  // every query is before every key or past the window of every key
  auto no_work = [&](int u) { return (32 * u + 31 < kbase) || (p.wl >= 0 && 32 * u > kbase + 16 * NKB - 1 + p.wl); };
  Walk cw = {0, rot0, 0};
  for (int k = 0; k < total;) {
    // G = 1: a step is a unit and its complement, of which a wave takes the one it has work in, or up to two units in a row.
    // G = 2: each group of waves has a unit of its own, alone or with its complement.
    const int prim = cw.u;
    const bool pair = prim < npair;
    advance(cw);
    int need = pair ? 2 : 1, next = -1;   // items of this step: k .. k + need - 1
    int u = prim, slot = G == 1 ? k : cslot;
    bool idle = false;
    if constexpr (G == 1) {
      if (!pair && k + 1 < total && cw.u >= npair) {
        next = cw.u;
        need = 2;
        advance(cw);
      }
    } else {
      const int n2 = k + need < total ? (cw.u < npair ? 2 : 1) : 0;
      const bool both = n2 && k + need + n2 <= issued;   // else the second group sits this step out
      if (grp) {
        idle = !both;
        u = cw.u;
        slot += need;
      }
      if (both) {
        need += n2;
        advance(cw);
      }
    }
    // they have landed (this wave's part; wave 0 carries one more load per item), then everybody's; the
    // requests after them stay in flight
    const int younger = issued - (k + need);
    if (wave == 0) wait_items<KV_LPW + 1, G>(younger);
    else wait_items<KV_LPW, G>(younger);
    lds_barrier();
    // every wave is past the items before k: their slots take the next requests
    for (; issued < total && issued < k + NR; ++issued) {
      if constexpr (G == 1) {
        issue_next(issued & (NR - 1));
      } else {
        issue_next(islot);
        islot = islot + 1 < NR ? islot + 1 : 0;
      }
    }
    if (u < npair && no_work(u)) {
      u += K0;
      ++slot;
    }
    k += need;
    if constexpr (G == 2) {
      slot = slot < NR ? slot : slot - NR;
      cslot = cslot + need < NR ? cslot + need : cslot + need - NR;
    }
    do {
      const uint32_t base = (uint32_t)((G == 1 ? slot & (NR - 1) : slot) * KV_ITEM);
      int lc = threadIdx.x & 63;
      asm volatile("" : "+v"(lc));
      const int l16 = lc & 15, kb = lc >> 4;
      kaddr = (uint32_t)((kb >> 1) * 512 + l16 * 32 + (kb & 1) * 16);
      vaddr = (uint32_t)((4 * kb + (l16 >> 2)) * 32 + 8 * (l16 & 3));
      faddr = vrows + (uint32_t)(lc * 16);
      if (!idle && !no_work(u)) {
        const bool edge = (32 * u < kbase + 16 * NKB - 1) || (p.wl >= 0 && 32 * u + 31 > kbase + p.wl) || (c0 + 32 * u + 32 > eos);
        // One stream of products: S = Q K^T, dP = dO V^T beside the exponentials of S, dV^T[d][key] += dO^T[d][q] P[q][key]
        // beside dS, dK^T[d][key] += Q^T[d][q] dS[q][key]; what a step multiplies was requested from LDS a step (1 KB row
        // fragments) or two (transposed ones) before.
        constexpr int PT = 2;       // transposed fragments are requested this many products ahead
        constexpr int NQ = 2 * NKB;   // quads of scores: (16-query block q & 1, 16-key block q >> 1)
        f32x4 S[NQ], dP[NQ];
        bf16x8 qa[KS][2], oa[KS][2], va[KS][NKB], ot[DB], qt[DB];
        // rows of the accumulators are the queries 16 qb + 4 kb + r, the column is this lane's key of its block; they start from
        // (-lse / scale, -delta) of their rows
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          qa[0][qb] = rfrag(base + KV_Q, qb, 0);
          const NHA_LDS f32x4* lp = reinterpret_cast<const NHA_LDS f32x4*>(lds + base + KV_LD + (16 * qb + 4 * kb) * 8);
          const f32x4 a0 = lp[0], a1 = lp[1];   // the pairs of rows r = 0, 1 and r = 2, 3
#pragma unroll
          for (int kk = 0; kk < NKB; ++kk) {
            S[qb + 2 * kk] = (f32x4){a0[0], a0[2], a1[0], a1[2]};
            dP[qb + 2 * kk] = (f32x4){a0[1], a0[3], a1[1], a1[3]};
          }
        }
        auto read_do = [&](int ks) {
#pragma unroll
          for (int qb = 0; qb < 2; ++qb) oa[ks][qb] = rfrag(base + KV_O, qb, ks);
#pragma unroll
          for (int kk = 0; kk < NKB; ++kk) va[ks][kk] = vfrag(kk, ks);
        };
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          __builtin_amdgcn_sched_barrier(0);
          if (ks + 1 < KS) {
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) qa[ks + 1][qb] = rfrag(base + KV_Q, qb, ks + 1);
          } else {
            read_do(0);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < NQ; ++q) S[q] = mfma16(qa[ks][q & 1], kfr[q >> 1][ks], S[q]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (edge) {
          const float none = cs < 0.f ? INFINITY : -INFINITY;   // -inf once it has been multiplied by cs below
#pragma unroll
          for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int y = 32 * u + 16 * (q & 1) + 4 * kb + r, xk = kbase + 16 * (q >> 1) + l16;
              const bool ok = (xk <= y) && (p.wl < 0 || y - xk <= p.wl) && (c0 + y < eos);
              if (!ok) S[q][r] = none;
            }
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          __builtin_amdgcn_sched_barrier(0);
          if (ks + 1 < KS) {
            read_do(ks + 1);
          } else {
#pragma unroll
            for (int i = 0; i < PT; ++i) ot[i] = tfrag(base + KV_O, i);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < NQ; ++q) dP[q] = mfma16(oa[ks][q & 1], va[ks][q >> 1], dP[q]);
          if (ks < NQ)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[ks][r] = fexp2(S[ks][r] * cs);
        }
        bf16x8 Pb[NKB], dSb[NKB];
#pragma unroll
        for (int kk = 0; kk < NKB; ++kk) Pb[kk] = pack8(S[2 * kk], S[2 * kk + 1]);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          __builtin_amdgcn_sched_barrier(0);
          if (db + PT < DB) ot[db + PT] = tfrag(base + KV_O, db + PT);
          else qt[db + PT - DB] = tfrag(base + KV_Q, db + PT - DB);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int kk = 0; kk < NKB; ++kk) dV[db][kk] = mfma16(ot[db], Pb[kk], dV[db][kk]);
          if (db >= 1 && db <= NQ) S[db - 1] *= dP[db - 1];
          if (db >= 1 && db <= NQ && db % 2 == 0) dSb[db / 2 - 1] = pack8(S[db - 2], S[db - 1]);
        }
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          __builtin_amdgcn_sched_barrier(0);
          if (db + PT < DB) qt[db + PT] = tfrag(base + KV_Q, db + PT);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int kk = 0; kk < NKB; ++kk) dK[db][kk] = mfma16(qt[db], dSb[kk], dK[db][kk]);
        }
      }
      u = next;
      next = -1;
      ++slot;
    } while (u >= 0);
  }
  // two groups: the second hands over dK, the first dV, a lane's sums at its own place in the memory of ring and V rows
  if (G == 2) {
    lds_barrier();
    NHA_LDS f32x4* const xk = (NHA_LDS f32x4*)lds + kw * (DB * NKB * 64) + lane;
    NHA_LDS f32x4* const xv = xk + KW * (DB * NKB * 64);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int kk = 0; kk < NKB; ++kk)
        if (grp) xk[(db * NKB + kk) * 64] = dK[db][kk];
        else xv[(db * NKB + kk) * 64] = dV[db][kk];
    lds_barrier();
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int kk = 0; kk < NKB; ++kk)
        if (grp) dV[db][kk] += xv[(db * NKB + kk) * 64];
        else dK[db][kk] += xk[(db * NKB + kk) * 64];
  }
#pragma unroll
  for (int kk = 0; kk < NKB; ++kk) {
    const int tk = c0 + kbase + 16 * kk + l16;
    if (tk >= eos) continue;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int64_t off = ((int64_t)tk * H + h) * D + 16 * db + 4 * kb;
      bf16x4 pk;
      if (G == 1 || !grp) {
#pragma unroll
        for (int r = 0; r < 4; ++r) pk[r] = (__bf16)(dK[db][kk][r] * p.scale);
        if constexpr (PARTS) *reinterpret_cast<f32x4*>(p.wk + blockIdx.z * p.pd + off) = dK[db][kk] * p.scale;
        else *reinterpret_cast<bf16x4*>(p.dk + off) = pk;
      }
      if (G == 1 || grp) {
        if constexpr (PARTS) {
          *reinterpret_cast<f32x4*>(p.wv + blockIdx.z * p.pd + off) = dV[db][kk];
          continue;
        }
        const float4 sv = *reinterpret_cast<const float4*>(p.dvs + off);
        pk[0] = (__bf16)(dV[db][kk][0] + sv.x);
        pk[1] = (__bf16)(dV[db][kk][1] + sv.y);
        pk[2] = (__bf16)(dV[db][kk][2] + sv.z);
        pk[3] = (__bf16)(dV[db][kk][3] + sv.w);
        *reinterpret_cast<bf16x4*>(p.dv + off) = pk;
      }
    }
  }
}

}  // namespace

// Served: four (or a multiple of four) query heads per kv-head at D = 128, tensors of one call below 4 GiB
// (32-bit lane offsets of the LDS-direct loads).
bool bwd_ring_supported(const NhaPrefillBwdArgs* a) {
#ifdef NHA_AB_SWITCHES   // measurement builds only (-DNHA_AB_SWITCHES)
  static const bool off = getenv("NHA_BWD_NO_RING") != nullptr;
#else
  constexpr bool off = false;
#endif
  if (off || a->K != 128 || a->V != 128 || a->HQ % a->H != 0 || (a->HQ / a->H) % 4 != 0) return false;
  return (int64_t)a->T_tot * a->HQ * 128 * 2 < ((int64_t)1 << 32);
}

static bool short_window(const NhaPrefillBwdArgs* a) { return a->wl >= 0 && a->wl < 160; }

// Parts of a kv-head's query heads: as many as all groups of 128 keys (at most) still have a place at once in (the scale is left out of it, as
// it is of a workspace's size).
int bwd_ring_dkv_parts(const NhaPrefillBwdArgs* a) {
  if (!bwd_ring_supported(a)) return 1;
  const int NG = a->HQ / a->H;
  const int64_t g128 = (int64_t)a->H * ((a->NT + a->N) / 2);
  int parts = 1;
  while (parts < 8 && NG % (2 * parts) == 0 && 2 * parts * g128 <= 256) parts *= 2;
  return parts;
}

// Keys per workgroup of the dk / dv kernel here, 0 where bwd_dkv_kernel takes the call.  Windows of less than 160 keys: 128.  Others: a
// workgroup of 128 keys takes 0.6 of the time of one of 256, so the fewer rounds of the 256 CUs decide.  us, 256 / 128 keys, 32 / 8
// heads: 5000 tokens, W = 512 (160 groups of 256 keys) 161 / 188, 2 x 5000 (320) W = 160 202 / 162, W = 300 241 / 220, W = 1000 467
// / 454, 3 x 4000 (384) W = 1000 520 / 483, 2 x 8192 (512) W = 512 373 / 422, W = 2048 1016 / 1262.
// The workgroup walks all queries that see its keys, whatever the size of the call; where even the groups of 128 fill half of the chip
// or less, the query heads are shared out (bwd_ring_dkv_parts), or, with many short sequences, bwd_dkv_kernel's groups of 64 take the
// call: us, bwd_dkv_kernel / this in parts and their sum, 32 / 4 heads: 525 packed tokens, W = 134 47 / 17, 2 x 533, W = 950 117 / 50,
// 2000, W = 300 86 / 46, 3500, W = 300 89 / 75, 4000, W = 500 131 / 102, 2969 packed, W = 70 51 / 41; 32 / 8, 2001, W = 200 44 / 42, 1500, W
// = 800 95 / 73; 8 / 2, 700, W = 100 29 / 16, 2778, W = 448 58 / 35, 4500, W = 300 48 / 43.
// Beyond, the groups of 64 pass one round of places and pull every q / do row twice as often: 2200 tokens, W = 200 (144) 65 / 59, W =
// 1000 183 / 160, 3000, W = 600 (192) 153 / 115, 4000, W = 1000 (256) 233 / 172, 8 / 2 heads, 4 x 4096, W = 512 132 / 105; short
// windows, 4000 tokens, W = 128 57 / 51.
// A scale of (almost) zero goes to bwd_dkv_kernel too: the scores here start from -lse / scale.
static int key_groups(const NhaPrefillBwdArgs* a) {
  if (!(fabsf(a->scale) > 1e-30f) || !bwd_ring_supported(a)) return 0;
  const int64_t g256 = (int64_t)a->H * ((a->NT + 3) / 4), g128 = (int64_t)a->H * ((a->NT + 1) / 2);
  if (g128 <= 128) return bwd_ring_dkv_parts(a) > 1 ? 128 : 0;
  if (short_window(a)) return 128;
  return (g128 + 255) / 256 * 6 < (g256 + 255) / 256 * 10 ? 128 : 256;
}

bool bwd_ring_dkv_supported(const NhaPrefillBwdArgs* a) {
  return key_groups(a) != 0;
}

int bwd_ring_dq(const NhaPrefillBwdArgs* a, const float* delta, float2* ld) {
  DqP p;
  p.q = (const bf16_t*)a->q_swa; p.k = (const bf16_t*)a->k_swa; p.v = (const bf16_t*)a->v; p.dout = (const bf16_t*)a->dout;
  p.lse_swa = a->lse_swa; p.lse_gsa = a->lse_gsa; p.delta = delta;
  p.dq = (bf16_t*)a->dq_swa; p.ld = ld;
  p.cu = a->cu_seqlens; p.cidx = a->chunk_indices;
  p.HQ = a->HQ; p.H = a->H; p.NG = a->HQ / a->H; p.NT = a->NT; p.wl = a->wl; p.scale = a->scale;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [&] {
    attr_err = hipFuncSetAttribute((const void*)ring_dq_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, BYTES);
    if (attr_err == hipSuccess) attr_err = hipFuncSetAttribute((const void*)ring_dq_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, BYTES);
  });
  if (attr_err != hipSuccess) {
    set_error("nha_prefill_bwd: cannot reserve %d bytes of LDS: %s", BYTES, hipGetErrorString(attr_err));
    return NHA_ERR_LAUNCH;
  }
  const dim3 grid(p.H * (p.NG / 4), p.NT);
  if (prefill_ring_raw(a->HQ, a->NT)) hipLaunchKernelGGL(ring_dq_kernel<true>, grid, dim3(512), BYTES, (hipStream_t)a->stream, p);
  else hipLaunchKernelGGL(ring_dq_kernel<false>, grid, dim3(512), BYTES, (hipStream_t)a->stream, p);
  NHA_CHECK_LAUNCH("nha_prefill_bwd(window dq, ring)");
  return NHA_OK;
}

int bwd_ring_dkv(const NhaPrefillBwdArgs* a, const float2* ld, const float* dvs, int parts, float* wk, float* wv) {
  DkvP p;
  p.q = (const bf16_t*)a->q_swa; p.k = (const bf16_t*)a->k_swa; p.v = (const bf16_t*)a->v; p.dout = (const bf16_t*)a->dout;
  p.ld = ld; p.dvs = dvs; p.wk = wk; p.wv = wv; p.pd = (int64_t)a->T_tot * a->H * a->K;
  p.dk = (bf16_t*)a->dk_swa; p.dv = (bf16_t*)a->dv;
  p.cu = a->cu_seqlens; p.cidx = a->chunk_indices;
  p.HQ = a->HQ; p.H = a->H; p.NG = a->HQ / a->H / parts; p.NT = a->NT; p.wl = a->wl; p.scale = a->scale;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [&] {
    auto reserve = [&](const void* kernel, int bytes) {
      if (attr_err == hipSuccess) attr_err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    };
    reserve((const void*)ring_dkv_kernel<256, 1, false>, KV_BYTES<256, 1>);
    reserve((const void*)ring_dkv_kernel<128, 1, false>, KV_BYTES<128, 1>);
    reserve((const void*)ring_dkv_kernel<128, 2, false>, KV_BYTES<128, 2>);
    reserve((const void*)ring_dkv_kernel<128, 1, true>, KV_BYTES<128, 1>);
    reserve((const void*)ring_dkv_kernel<128, 2, true>, KV_BYTES<128, 2>);
  });
  if (attr_err != hipSuccess) {
    set_error("nha_prefill_bwd: cannot reserve %d bytes of LDS: %s", KV_BYTES<256, 1>, hipGetErrorString(attr_err));
    return NHA_ERR_LAUNCH;
  }
  // one launch row per chunk, rounded up to whole key groups (4 chunks of 256 keys, 2 of 128)
  const dim3 halves(p.H, 2 * ((p.NT + 1) / 2), parts);
  hipStream_t st = (hipStream_t)a->stream;
  if (key_groups(a) == 256)
    hipLaunchKernelGGL((ring_dkv_kernel<256, 1, false>), dim3(p.H, 4 * ((p.NT + 3) / 4)), dim3(512), (KV_BYTES<256, 1>), st, p);
  else if (short_window(a) && parts > 1)
    hipLaunchKernelGGL((ring_dkv_kernel<128, 1, true>), halves, dim3(512), (KV_BYTES<128, 1>), st, p);
  else if (short_window(a))
    hipLaunchKernelGGL((ring_dkv_kernel<128, 1, false>), halves, dim3(512), (KV_BYTES<128, 1>), st, p);
  else if (parts > 1)
    hipLaunchKernelGGL((ring_dkv_kernel<128, 2, true>), halves, dim3(512), (KV_BYTES<128, 2>), st, p);
  else
    hipLaunchKernelGGL((ring_dkv_kernel<128, 2, false>), halves, dim3(512), (KV_BYTES<128, 2>), st, p);
  NHA_CHECK_LAUNCH("nha_prefill_bwd(window dk, dv, ring)");
  return NHA_OK;
}

}  // namespace nha
