// Matrix-core kernels for the window branch of the NHA prefill backward on gfx950
// (bf16, K == V == D in {64,128,256}; the part nha_fla/ops/nha/chunk.py:499-511 hands to
// flash-attn's backward).  With the merged-softmax quantities of the whole op per (token, q-head)
//   lse = log(sum_m e^u + sum_j e^w),   delta = do . o,
// the window logits w[q][j] = scale q_swa_q . k_swa_j (j in [max(bos, q - wl), q]) give
//   pi = e^(w - lse),  dpi = do_q . v_j,  dw = pi (dpi - delta),
//   dq_swa_q = scale sum_j dw k_swa_j,   dk_swa_j = scale sum_q dw q_swa_q,   dv_j += sum_q pi do_q.
// Two kernels, for what prefill_bwd_ring.hip and prefill_bwd_ring256.hip do not take, each in the orientation whose
// accumulator layout feeds its next MFMA without moving data between lanes (v_mfma_f32_16x16x32_bf16: A[i][8(l/16)+e],
// B[8(l/16)+e][j], C[4(l/16)+r][l%16]):
//   bwd_dq_kernel   one workgroup per (64 queries, q-head); K/V tiles stream through LDS;
//                   S^T = K Q^T and dP^T = V dO^T put a query per lane, dQ^T += K^T dS^T
//   bwd_dkv_kernel  one workgroup per (64 keys, kv-head); Q/dO tiles of every q-head of the group
//                   stream through LDS; S = Q K^T and dP = dO V^T put a key per lane,
//                   dV^T += dO^T P and dK^T += Q^T dS
#include "common.h"

namespace nha {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
#define NHA_LDS __attribute__((address_space(3)))
typedef NHA_LDS bf16_t lbf16;
typedef NHA_LDS float lfloat;

constexpr int BT = 64;
constexpr float LOG2E = 1.4426950408889634f;

struct WP {
  const bf16_t *q, *k, *v, *dout;          // q_swa [T,HQ,D]; k_swa, v [T,H,D]; dout [T,HQ,D]
  const float *lse_swa, *lse_gsa, *delta;  // [T,HQ]
  const float* dvs;                        // [T,H,D] slot-branch part of dv
  float2* ld;                              // [T,HQ] out of the dq kernel, where the dk / dv kernel wants it: (-lse log2(e), -delta)
  bf16_t *dq, *dk, *dv;
  const int32_t *cu, *cidx;
  int HQ, H, NG, wl;
  float scale;
};

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ void lds_st16(lbf16* p, uint4 v) { *reinterpret_cast<NHA_LDS u32x4*>(p) = (u32x4){v.x, v.y, v.z, v.w}; }
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ bf16x8 pack8(f32x4 a, f32x4 b) {
  bf16x8 r;
  r[0] = (__bf16)a[0]; r[1] = (__bf16)a[1]; r[2] = (__bf16)a[2]; r[3] = (__bf16)a[3];
  r[4] = (__bf16)b[0]; r[5] = (__bf16)b[1]; r[6] = (__bf16)b[2]; r[7] = (__bf16)b[3];
  return r;
}
// 8 consecutive elements of row `row` of a row-major LDS tile, starting at `col`
__device__ __forceinline__ bf16x8 lds_frag(const lbf16* tile, int ld, int row, int col) {
  return *reinterpret_cast<const NHA_LDS bf16x8*>(tile + row * ld + col);
}
// transposed fragment: lane (c = l%16, kb = l/16) receives X[r0a + 4 kb + e][col0 + c], e = 0..3,
// and X[r0b + 4 kb + e][col0 + c] as elements 4..7
__device__ __forceinline__ bf16x8 lds_frag_tr(const lbf16* tile, int ld, int r0a, int r0b, int col0, int lane) {
  const int l16 = lane & 15, kb = lane >> 4;
  const lbf16* pa = tile + (r0a + 4 * kb + (l16 >> 2)) * ld + col0 + 4 * (l16 & 3);
  const lbf16* pb = tile + (r0b + 4 * kb + (l16 >> 2)) * ld + col0 + 4 * (l16 & 3);
  struct { s16x4 a, b; } t;
  t.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pa);
  t.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pb);
  return __builtin_bit_cast(bf16x8, t);
}
// Query head of workgroup x in a launch whose rows hold one workgroup per query head.  Workgroups are dealt
// to the 8 XCDs in launch order, so x runs on XCD x % 8: the heads are numbered so that an XCD gets
// consecutive heads, and the query heads of one kv-head fetch its states and rows through one L2.
__device__ __forceinline__ int head_of_workgroup(int x, int HQ) { return (HQ & 7) == 0 ? (x & 7) * (HQ >> 3) + (x >> 3) : x; }
// (head, row of the launch) of a workgroup of the window kernels, grid (heads, chunks).  With 8 heads or a multiple
// the launch order already keeps a head on one XCD (head_of_workgroup).  With fewer -- the 340M layers have four -- the
// chunks of a head would alternate between XCDs (workgroup L runs on XCD L % 8 and L = row * heads + head), and the
// window rows that neighbouring chunks share would be fetched into two L2s, each holding twice the span of chunks:
// there XCD k takes the k-th eighth of the (head, row) sequence, consecutive rows of one head.
__device__ __forceinline__ void window_tile(int heads, int& head, int& row) {
  const int total = gridDim.x * gridDim.y;
  if ((heads & 7) == 0) {
    head = head_of_workgroup(blockIdx.x, heads);
    row = blockIdx.y;
  } else {
    // the first 8 * (total / 8) workgroups are dealt as said, the up to seven left over keep their place
    const int L = blockIdx.y * gridDim.x + blockIdx.x, per = total >> 3;
    const int v = L < 8 * per ? (L & 7) * per + (L >> 3) : L;
    head = v / (int)gridDim.y;
    row = v % (int)gridDim.y;
  }
}
__device__ __forceinline__ float logaddexp_f(float a, float b) {
  const float mx = fmaxf(a, b);
  return mx + logf(expf(a - mx) + expf(b - mx));
}

// rows [0, vhi) of a ROWS x D tile whose row r is global row grow0 + r of a [*, heads, D] tensor
template <int ROWS, int D, int THREADS = 256>
struct Tile {
  static constexpr int NPC = ROWS * D / 8 / THREADS;
  uint4 r[NPC];
  __device__ __forceinline__ void load(const bf16_t* base, int64_t row_stride, int64_t grow0, int vhi, int tid) {
#pragma unroll
    for (int u = 0; u < NPC; ++u) {
      const int c = tid + THREADS * u;
      const int row = c / (D / 8), col = (c % (D / 8)) * 8;
      uint4 x = make_uint4(0, 0, 0, 0);
      if (row < vhi) x = *reinterpret_cast<const uint4*>(base + (grow0 + row) * row_stride + col);
      r[u] = x;
    }
  }
  __device__ __forceinline__ void store(lbf16* lds, int tid) const {
#pragma unroll
    for (int u = 0; u < NPC; ++u) {
      const int c = tid + THREADS * u;
      const int row = c / (D / 8), col = (c % (D / 8)) * 8;
      lds_st16(lds + row * (D + 16) + col, r[u]);
    }
  }
};

// ------------------------------------------------------------------------------------------
// dq_swa: grid (HQ, NT), 4 waves x 16 query rows
// ------------------------------------------------------------------------------------------
template <int D, int TK>
__global__ __launch_bounds__(256) void bwd_dq_kernel(const WP p) {
  constexpr int KS = D / 32, DB = D / 16, LDT = D + 16, NH = TK / 32, TILE = TK * LDT;
  extern __shared__ __align__(16) unsigned char smem[];
  lbf16* const tiles = (lbf16*)smem;   // K0, K1, V0, V1
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, kb = lane >> 4;
  const int H = p.H, HQ = p.HQ;
  int hq, wrow;
  window_tile(p.HQ, hq, wrow);
  const int h = hq / p.NG;
  // last chunk first: the chunks at the start of a sequence see the fewest keys, and short
  // workgroups at the end of the launch leave the smallest tail
  const int chunk = gridDim.y - 1 - wrow;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int c0 = bos + it * BT;
  const int rows = (eos - c0) < BT ? (eos - c0) : BT;
  const int y = 16 * wave + l16;   // this lane's query, relative to the chunk
  const bool valid = y < rows;
  const int64_t tq = (int64_t)(c0 + (valid ? y : 0)) * HQ + hq;
  bf16x8 qf[KS], df[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    uint4 a = make_uint4(0, 0, 0, 0), b = a;
    if (valid) {
      a = *reinterpret_cast<const uint4*>(p.q + tq * D + 32 * ks + 8 * kb);
      b = *reinterpret_cast<const uint4*>(p.dout + tq * D + 32 * ks + 8 * kb);
    }
    qf[ks] = __builtin_bit_cast(bf16x8, a);
    df[ks] = __builtin_bit_cast(bf16x8, b);
  }
  const float lse2 = valid ? logaddexp_f(p.lse_swa[tq], p.lse_gsa[tq]) * LOG2E : 0.f;
  const float dl = valid ? p.delta[tq] : 0.f;
  const float cs = p.scale * LOG2E;
  if (p.ld && valid && kb == 0) p.ld[tq] = make_float2(-lse2, -dl);
  f32x4 dQ[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dQ[db] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // key tile i covers keys [c0 + 64 - TK (i+1), c0 + 64 - TK i); boundaries are multiples of TK
  // away from bos, so no tile starts before its sequence
  int lowest = bos;
  if (p.wl >= 0 && c0 - p.wl > bos) lowest = c0 - p.wl;
  const int ntiles = (c0 + 64 - lowest + TK - 1) / TK;
  Tile<TK, D> rk, rv;
  auto issue = [&](int i) {
    const int64_t grow0 = (int64_t)c0 + 64 - TK * (i + 1);
    int vhi = eos - (int)grow0;
    vhi = vhi < 0 ? 0 : (vhi > TK ? TK : vhi);
    rk.load(p.k + (int64_t)h * D, (int64_t)H * D, grow0, vhi, tid);
    rv.load(p.v + (int64_t)h * D, (int64_t)H * D, grow0, vhi, tid);
  };
  issue(0);
  rk.store(tiles, tid);
  rv.store(tiles + 2 * TILE, tid);
  if (ntiles > 1) issue(1);
  lds_barrier();
  for (int i = 0; i < ntiles; ++i) {
    const int cur = i & 1;
    const lbf16* Kt = tiles + cur * TILE;
    const lbf16* Vt = tiles + (2 + cur) * TILE;
    const int xbase = 64 - TK * (i + 1);
    const bool edge = (xbase + TK - 1 > 0) || (p.wl >= 0 && p.wl < TK * (i + 1) - 1);
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) {
      f32x4 S[2], dP[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        S[kk] = (f32x4){0.f, 0.f, 0.f, 0.f};
        dP[kk] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          S[kk] = mfma16(lds_frag(Kt, LDT, 32 * hf + 16 * kk + l16, 32 * ks + 8 * kb), qf[ks], S[kk]);
          dP[kk] = mfma16(lds_frag(Vt, LDT, 32 * hf + 16 * kk + l16, 32 * ks + 8 * kb), df[ks], dP[kk]);
        }
      }
      f32x4 dS[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int x = xbase + 32 * hf + 16 * kk + 4 * kb + r;
          const bool ok = !edge || ((x <= y) && (p.wl < 0 || x >= y - p.wl));
          const float pr = ok ? fexp2(S[kk][r] * cs - lse2) : 0.f;
          dS[kk][r] = pr * (dP[kk][r] - dl) * p.scale;
        }
      const bf16x8 dSb = pack8(dS[0], dS[1]);
      // dQ^T[d][q] += K^T[d][key] dS^T[key][q]
#pragma unroll
      for (int db = 0; db < DB; ++db) dQ[db] = mfma16(lds_frag_tr(Kt, LDT, 32 * hf, 32 * hf + 16, 16 * db, lane), dSb, dQ[db]);
    }
    if (i + 1 < ntiles) {
      rk.store(tiles + (cur ^ 1) * TILE, tid);
      rv.store(tiles + (2 + (cur ^ 1)) * TILE, tid);
      if (i + 2 < ntiles) issue(i + 2);
    }
    lds_barrier();
  }
  if (valid) {
    bf16_t* op = p.dq + tq * D + 4 * kb;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      bf16x4 pk;
#pragma unroll
      for (int r = 0; r < 4; ++r) pk[r] = (__bf16)dQ[db][r];
      *reinterpret_cast<bf16x4*>(op + 16 * db) = pk;
    }
  }
}

// ------------------------------------------------------------------------------------------
// dk_swa, dv: grid (H, NT), 4 waves x 16 keys.  MODE 0: both; 1: dk only; 2: dv only (D = 256: both accumulators do not
// fit the register file, and the workgroups of one launch (SPLIT) take 1 or 2; as two launches a small call ran each on
// half of the chip: 1700 tokens, 4 heads 50 -> 26 us; 8 x 2048 tokens 217 -> 201 us)
// G = 2: eight waves, every tile's queries halved between two groups of four, whose sums are added at the end.  A step of
// one wave per SIMD is a chain of LDS reads, products and exponentials (2.8 us for 64 x 64 scores at D = 128, whose products
// take 0.4); where a call has no second workgroup for the CU the second group fills the gaps: 1.9 us, 2001 packed tokens, 32 / 8
// heads, W = 571 114 -> 79 us.  Past that LDS itself bounds the step: each wave reads both tiles for its 16 keys.
// ------------------------------------------------------------------------------------------
template <int D, int TQ, int MODE, int G>
__device__ __forceinline__ void bwd_dkv_tile(const WP& p) {
  constexpr int KS = D / 32, DB = D / 16, LDT = D + 16, NH = TQ / 32 / G, TILE = TQ * LDT;
  constexpr bool DO_K = MODE != 2, DO_V = MODE != 1;
  extern __shared__ __align__(16) unsigned char smem[];
  lbf16* const tiles = (lbf16*)smem;                 // Q0, Q1, dO0, dO1
  lfloat* const lsb = (lfloat*)(tiles + 4 * TILE);   // [2][TQ] lse * log2(e)
  lfloat* const dlb = lsb + 2 * TQ;                  // [2][TQ] delta
  const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) & 3;
  const int hf0 = G == 1 ? 0 : NH * (tid >> 8);   // first block of 32 queries of this group of waves
  const int l16 = lane & 15, kb = lane >> 4;
  const int H = p.H, HQ = p.HQ, NG = p.NG;
  int h, chunk;
  window_tile(H, h, chunk);
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int j0 = bos + it * BT;
  const int krows = (eos - j0) < BT ? (eos - j0) : BT;
  const int x = 16 * wave + l16;   // this lane's key, relative to j0
  const bool valid = x < krows;
  const int64_t jk = (int64_t)(j0 + (valid ? x : 0)) * H + h;
  bf16x8 kf[KS], vf[DO_K ? KS : 1];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    uint4 a = make_uint4(0, 0, 0, 0), b = a;
    if (valid) {
      a = *reinterpret_cast<const uint4*>(p.k + jk * D + 32 * ks + 8 * kb);
      if (DO_K) b = *reinterpret_cast<const uint4*>(p.v + jk * D + 32 * ks + 8 * kb);
    }
    kf[ks] = __builtin_bit_cast(bf16x8, a);
    if (DO_K) vf[ks] = __builtin_bit_cast(bf16x8, b);
  }
  const float cs = p.scale * LOG2E;
  f32x4 dK[DO_K ? DB : 1], dV[DO_V ? DB : 1];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    if (DO_K) dK[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (DO_V) dV[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  // queries that see any of these keys: [j0, qend); tiles of TQ queries x the NG heads of the group
  int qend = eos;
  if (p.wl >= 0 && j0 + 64 + p.wl < eos) qend = j0 + 64 + p.wl;
  const int nqt = (qend - j0 + TQ - 1) / TQ;
  const int niter = nqt * NG;
  Tile<TQ, D, 256 * G> rq, ro;
  float rls = 0.f, rlg = 0.f, rd = 0.f;
  // iteration i = (q-head of the group, query tile), tiles innermost: the workgroup of the next
  // chunk (same XCD, started together) reads the same tile one iteration earlier, so the tile is
  // still in that XCD's L2; with the heads innermost the reuse distance was four iterations of
  // every resident workgroup, more than the L2 holds.
  auto issue = [&](int i) {
    const int qt = i % nqt, hq = h * NG + i / nqt;
    const int64_t grow0 = (int64_t)j0 + TQ * qt;
    int vhi = eos - (int)grow0;
    vhi = vhi < 0 ? 0 : (vhi > TQ ? TQ : vhi);
    rq.load(p.q + (int64_t)hq * D, (int64_t)HQ * D, grow0, vhi, tid);
    ro.load(p.dout + (int64_t)hq * D, (int64_t)HQ * D, grow0, vhi, tid);
    // only requested here: the merge of the two log-sum-exps waits until the values are staged, a
    // tile later (used at once, it stalled the first wave for a memory latency in every iteration
    // and the other waves behind it at the barrier)
    rls = rlg = rd = 0.f;
    if (tid < TQ && tid < vhi) {
      const int64_t tq = (grow0 + tid) * HQ + hq;
      rls = p.lse_swa[tq];
      rlg = p.lse_gsa[tq];
      rd = p.delta[tq];
    }
  };
  auto stage = [&](int buf) {
    rq.store(tiles + buf * TILE, tid);
    ro.store(tiles + (2 + buf) * TILE, tid);
    if (tid < TQ) {
      lsb[buf * TQ + tid] = logaddexp_f(rls, rlg) * LOG2E;
      dlb[buf * TQ + tid] = rd;
    }
  };
  issue(0);
  stage(0);
  if (niter > 1) issue(1);
  lds_barrier();
  for (int i = 0; i < niter; ++i) {
    const int cur = i & 1;
    const lbf16* Qt = tiles + cur * TILE;
    const lbf16* Ot = tiles + (2 + cur) * TILE;
    const lfloat* ls = lsb + cur * TQ;
    const lfloat* dl = dlb + cur * TQ;
    const int ybase = TQ * (i % nqt);   // first query of the tile, relative to j0
    const bool edge = (ybase < 63) || (p.wl >= 0 && ybase + TQ - 1 > p.wl) || (j0 + ybase + TQ > eos);
#pragma unroll
    for (int hh = 0; hh < NH; ++hh) {
      const int hf = hf0 + hh;
      f32x4 S[2], dP[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        S[kk] = (f32x4){0.f, 0.f, 0.f, 0.f};
        dP[kk] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
      // the fragments of a 16-query block are requested together, then multiplied: one LDS
      // latency per block instead of one per MFMA
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        constexpr int KH = KS > 4 ? 4 : KS;   // fragments in flight per tensor
#pragma unroll
        for (int k0 = 0; k0 < KS; k0 += KH) {
          bf16x8 qa[KH], oa[DO_K ? KH : 1];
#pragma unroll
          for (int u = 0; u < KH; ++u) {
            qa[u] = lds_frag(Qt, LDT, 32 * hf + 16 * kk + l16, 32 * (k0 + u) + 8 * kb);
            if (DO_K) oa[u] = lds_frag(Ot, LDT, 32 * hf + 16 * kk + l16, 32 * (k0 + u) + 8 * kb);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int u = 0; u < KH; ++u) {
            S[kk] = mfma16(qa[u], kf[k0 + u], S[kk]);
            if (DO_K) dP[kk] = mfma16(oa[u], vf[k0 + u], dP[kk]);
          }
        }
      }
      f32x4 P[2], dS[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int yr0 = 32 * hf + 16 * kk + 4 * kb;   // first of this lane's 4 query rows in the tile
        const f32x4 l4 = *reinterpret_cast<const NHA_LDS f32x4*>(ls + yr0);
        const f32x4 d4 = *reinterpret_cast<const NHA_LDS f32x4*>(dl + yr0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int yy = ybase + yr0 + r;
          const bool ok = !edge || ((x <= yy) && (p.wl < 0 || x >= yy - p.wl) && (j0 + yy < eos));
          const float pr = ok ? fexp2(S[kk][r] * cs - l4[r]) : 0.f;
          P[kk][r] = pr;
          dS[kk][r] = pr * (dP[kk][r] - d4[r]) * p.scale;
        }
      }
      const bf16x8 Pb = pack8(P[0], P[1]);
      const bf16x8 dSb = pack8(dS[0], dS[1]);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        // dV^T[d][key] += dO^T[d][q] P[q][key];  dK^T[d][key] += Q^T[d][q] dS[q][key]
        if (DO_V) dV[db] = mfma16(lds_frag_tr(Ot, LDT, 32 * hf, 32 * hf + 16, 16 * db, lane), Pb, dV[db]);
        if (DO_K) dK[db] = mfma16(lds_frag_tr(Qt, LDT, 32 * hf, 32 * hf + 16, 16 * db, lane), dSb, dK[db]);
      }
    }
    if (i + 1 < niter) {
      stage(cur ^ 1);
      if (i + 2 < niter) issue(i + 2);
    }
    lds_barrier();
  }
  if constexpr (G == 2) {
    // The two groups of waves have each summed one half of every tile's queries: the second hands over dK, the first dV (with
    // one of the two here, the second hands that over), a lane's sums at its own place in the tiles' memory.
    NHA_LDS f32x4* const xk = (NHA_LDS f32x4*)smem + (wave * DB) * 64 + lane;
    NHA_LDS f32x4* const xv = xk + (MODE == 0 ? 4 * DB * 64 : 0);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if (DO_K && hf0) xk[db * 64] = dK[db];
      if (DO_V && (MODE == 2 ? hf0 != 0 : hf0 == 0)) xv[db * 64] = dV[db];
    }
    lds_barrier();
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if (DO_K && !hf0) dK[db] += xk[db * 64];
      if (DO_V && (MODE == 2 ? hf0 == 0 : hf0 != 0)) dV[db] += xv[db * 64];
    }
  }
  const bool out_k = G == 1 || hf0 == 0, out_v = G == 1 || (MODE == 2 ? hf0 == 0 : hf0 != 0);
  if (valid) {
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int64_t off = jk * D + 16 * db + 4 * kb;
      bf16x4 pk;
      if (DO_K && out_k) {
#pragma unroll
        for (int r = 0; r < 4; ++r) pk[r] = (__bf16)dK[db][r];
        *reinterpret_cast<bf16x4*>(p.dk + off) = pk;
      }
      if (DO_V && out_v) {
        const float4 sv = *reinterpret_cast<const float4*>(p.dvs + off);
        pk[0] = (__bf16)(dV[db][0] + sv.x);
        pk[1] = (__bf16)(dV[db][1] + sv.y);
        pk[2] = (__bf16)(dV[db][2] + sv.z);
        pk[3] = (__bf16)(dV[db][3] + sv.w);
        *reinterpret_cast<bf16x4*>(p.dv + off) = pk;
      }
    }
  }
}

template <int D, int TQ, bool SPLIT, int G>
__global__ __launch_bounds__(256 * G) void bwd_dkv_kernel(const WP p) {
  if constexpr (SPLIT) {
    if (blockIdx.z == 0) bwd_dkv_tile<D, TQ, 1, G>(p);
    else bwd_dkv_tile<D, TQ, 2, G>(p);
  } else {
    bwd_dkv_tile<D, TQ, 0, G>(p);
  }
}


// ------------------------------------------------------------------------------------------
// Slot branch, the parts that involve the state gradient carried in from later chunks (the rest: prefill_bwd_slot.hip)
// ------------------------------------------------------------------------------------------
// bf16 row stride of tables of 64 columns in LDS.  They are read 16 bytes per lane of 16 rows and transposed: 4.15 and 3.3
// cycles per wave instruction at 80 (a workgroup of eight waves), 8.1 and 4.4 at 72.
constexpr int TLD = 80;

struct SP2 {
  const bf16_t *kg, *v, *s;          // k_gsa, v [T,H,D]; s [T,H,64]
  const float* gc;                   // [NT][H][64][64] gate cumsums (rows past the chunk's end repeat the last)
  const float *ek, *ev;              // [NT][H][D][64] x2
  const float* dks;                  // [T][H][D] intra-chunk part of dk_gsa (source-token index)
  float* dvs;                        // the same of the slot-branch dv; completed here
  const float* xg;                   // [T][H][64] first part of the dg summand
  float *dsi, *gtot;                 // [T][H][64] intra-chunk part of ds, then the chunk's reverse cumulative sums; [NT][H][64] their totals
  bf16_t* ds;                        // [T,H,64]
  bf16_t* dkg;                       // dk_gsa [T,H,D]
  const int32_t *cu, *cidx;
  int H, shift;
};

// x as a bf16 pair hi + lo (16 mantissa bits): the tables built from fp32 intermediates are kept
// this way and multiplied as hi*b + lo*b, so that their rounding stays below that of the bf16 inputs.
// Four consecutive elements at once: two 8-byte LDS writes (idx a multiple of 4)
__device__ __forceinline__ void split4_bf16(const float4 x, lbf16* hi, lbf16* lo, int idx) {
  const float v[4] = {x.x, x.y, x.z, x.w};
  bf16x4 h, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    h[e] = (__bf16)v[e];
    l[e] = (__bf16)(v[e] - (float)h[e]);
  }
  *reinterpret_cast<NHA_LDS bf16x4*>(hi + idx) = h;
  *reinterpret_cast<NHA_LDS bf16x4*>(lo + idx) = l;
}

// bwd_slot_inter_kernel, grid (H, NT): the parts that involve E_c, the state gradient carried
// into the END of chunk c (z even: k-state, rows k', output dk_gsa; z odd: v-state, rows v', output
// dvs), with dec_r[m] = e^(gl[m] - gc_r[m]):
//   out[r][x] = intra part + sum_m (s_r[m] dec_r[m]) E[x][m]         as out^T = E sE^T
//   ds[r][m] += dec_r[m] sum_x y_r[x] E[x][m]                         as Y E
// z / 2 picks DW of the D columns x: at head size 256 a part of half the columns leaves room for two workgroups on a CU.
// A workgroup takes the parts of its chunk one after the other (the next one's operands requested during the products), keeps
// their sums for ds, and goes on with the gates: ds complete, and the chunk's reverse cumulative sums of the dg summand
// xg - s ds with their total.  Bound: HBM.  With a workgroup per part, the sums handed on through memory and the gates in a
// launch of their own: B=2, T=8192, 32/8 heads of 128 98 + 31 -> 93 us; B=8, T=2048, 4 heads of 256 119 + 28 -> 98; 5003 packed
// tokens, 16 heads of 64 44 + 22 -> 44; 300 tokens, 4 heads of 256 (20 workgroups in place of 80) 20.5 -> 19.6 together.
template <int D, int DW>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void bwd_slot_inter_kernel(const SP2 p) {
  constexpr int DB = DW / 16, LDT = DW + 16, TILE = BT * LDT, ELD = TLD, NH = D / DW, NZ = 2 * NH;
  constexpr int NY = BT * DW / 8 / 256, NE = DW * BT / 4 / 256, NS = BT * BT / 4 / 256;
  extern __shared__ __align__(16) unsigned char smem[];
  lbf16* const Yt = (lbf16*)smem;        // [64 rows r][DW]  k' / v'
  lbf16* const Et = Yt + TILE;           // [DW x][ELD]      E[x][m], high part
  lbf16* const El = Et + DW * ELD;       //                  low part
  lbf16* const St = El + DW * ELD;        // [64 r][TLD]      s_r[m] dec_r[m], high part
  lbf16* const Sl = St + BT * TLD;       //                  low part
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, kb = lane >> 4;
  const int H = p.H;
  const int h = blockIdx.x, chunk = blockIdx.y;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int c0 = bos + it * BT;
  const int R = (eos - c0) < BT ? (eos - c0) : BT;
  int vlo = p.shift - it * BT;
  vlo = vlo < 0 ? 0 : vlo;
  const float* const gcb = p.gc + ((int64_t)chunk * H + h) * BT * BT;
  struct Part {
    uint4 y[NY];
    float4 e[NE];
  };
  auto request = [&](Part& t, int z) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // addresses derived anew for every part: there are no registers to keep them
    const bool isv = (z & 1) != 0;
    const int x0 = (z >> 1) * DW;
    const bf16_t* const ysrc = isv ? p.v : p.kg;
#pragma unroll
    for (int u = 0; u < NY; ++u) {
      const int c = tid + 256 * u;
      const int row = c / (DW / 8), cc = (c % (DW / 8)) * 8;
      t.y[u] = make_uint4(0, 0, 0, 0);
      if (row >= vlo && row < R) t.y[u] = *reinterpret_cast<const uint4*>(ysrc + (((int64_t)c0 + row - p.shift) * H + h) * D + x0 + cc);
    }
    const float4* const ep4 = reinterpret_cast<const float4*>((isv ? p.ev : p.ek) + (((int64_t)chunk * H + h) * D + x0) * BT);
#pragma unroll
    for (int u = 0; u < NE; ++u) t.e[u] = ep4[tid + 256 * u];
  };
  auto place = [&](const Part& t) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
#pragma unroll
    for (int u = 0; u < NY; ++u) {
      const int c = tid + 256 * u;
      lds_st16(Yt + c / (DW / 8) * LDT + (c % (DW / 8)) * 8, t.y[u]);
    }
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      const int e = 4 * (tid + 256 * u);
      split4_bf16(t.e[u], Et, El, (e >> 6) * ELD + (e & 63));
    }
  };
  Part part;
  request(part, 0);
  {
    float4 gl[NS], gr[NS];
    uint2 sr[NS];
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      const int e = 4 * (tid + 256 * u), r = e >> 6, m = e & 63;
      gl[u] = gr[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      sr[u] = make_uint2(0, 0);
      if (r >= vlo && r < R) {
        sr[u] = *reinterpret_cast<const uint2*>(p.s + (((int64_t)c0 + r - p.shift) * H + h) * BT + m);
        gl[u] = *reinterpret_cast<const float4*>(gcb + (BT - 1) * BT + m);
        gr[u] = *reinterpret_cast<const float4*>(gcb + r * BT + m);
      }
    }
    place(part);
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      const int e = 4 * (tid + 256 * u), r = e >> 6, m = e & 63;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (r >= vlo && r < R) {
        v.x = __uint_as_float(sr[u].x << 16) * __expf(gl[u].x - gr[u].x);
        v.y = __uint_as_float(sr[u].x & 0xffff0000u) * __expf(gl[u].y - gr[u].y);
        v.z = __uint_as_float(sr[u].y << 16) * __expf(gl[u].z - gr[u].z);
        v.w = __uint_as_float(sr[u].y & 0xffff0000u) * __expf(gl[u].w - gr[u].w);
      }
      split4_bf16(v, St, Sl, r * TLD + m);
    }
  }
  lds_barrier();
  const int col = 16 * wave + l16;
  // the gates' own rows: four consecutive rows 4 rg + q, four slots gm ..; and the gate rows of the decay of ds
  const int rg = tid >> 4, gm = (tid & 15) * 4;
  float4 gi[4], gx[4];
  uint2 gsv[4];
  float glast, grow[4][4];
  auto request_gates = [&]() {
    glast = gcb[(BT - 1) * BT + col];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int q = 0; q < 4; ++q) grow[rb][q] = gcb[(16 * rb + 4 * kb + q) * BT + col];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = 4 * rg + q;
      gi[q] = gx[q] = make_float4(0.f, 0.f, 0.f, 0.f);
      gsv[q] = make_uint2(0, 0);
      if (r >= vlo && r < R) {
        const int64_t rt = (((int64_t)c0 + r) * H + h) * BT + gm;
        gi[q] = *reinterpret_cast<const float4*>(p.dsi + rt);
        gx[q] = *reinterpret_cast<const float4*>(p.xg + rt);
        gsv[q] = *reinterpret_cast<const uint2*>(p.s + (((int64_t)c0 + r - p.shift) * H + h) * BT + gm);
      }
    }
  };
  const bool has = col >= vlo && col < R;
  f32x4 dsa[4];   // ds / dec: rows r = 16 rb + 4 kb + q, slot col
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) dsa[rb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int z = 0; z < NZ; ++z) {
    const bool isv = (z & 1) != 0;
    const int64_t oi = (((int64_t)c0 + col - p.shift) * H + h) * D + (z >> 1) * DW;
    // the partial sums the first products are added to, then the next part's operands: requested before the products
    const float* const old = isv ? p.dvs : p.dks;
    float4 pve[DB];
    if (has) {
#pragma unroll
      for (int db = 0; db < DB; ++db) pve[db] = *reinterpret_cast<const float4*>(old + oi + 16 * db + 4 * kb);
    }
    if (z + 1 < NZ) request(part, z + 1);
    else request_gates();
    // out^T[x][r = col] = sum_m E[x][m] sE[r][m]: A = E rows (plain), B = sE rows (plain), contraction m in 2 steps
    f32x4 accO[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) accO[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const bf16x8 bs = lds_frag(St, TLD, col, 32 * ks + 8 * kb), bsl = lds_frag(Sl, TLD, col, 32 * ks + 8 * kb);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const bf16x8 eh = lds_frag(Et, ELD, 16 * db + l16, 32 * ks + 8 * kb);
        accO[db] = mfma16(eh, bs, mfma16(eh, bsl, mfma16(lds_frag(El, ELD, 16 * db + l16, 32 * ks + 8 * kb), bs, accO[db])));
      }
    }
    if (has) {
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const float o0 = accO[db][0] + pve[db].x, o1 = accO[db][1] + pve[db].y, o2 = accO[db][2] + pve[db].z, o3 = accO[db][3] + pve[db].w;
        if (isv) {
          *reinterpret_cast<float4*>(p.dvs + oi + 16 * db + 4 * kb) = make_float4(o0, o1, o2, o3);
        } else {
          bf16x4 pk;
          pk[0] = (__bf16)o0; pk[1] = (__bf16)o1; pk[2] = (__bf16)o2; pk[3] = (__bf16)o3;
          *reinterpret_cast<bf16x4*>(p.dkg + oi + 16 * db + 4 * kb) = pk;
        }
      }
    }
    // ds[r][m = col] / dec += sum_x y_r[x] E[x][m]: A = y rows (two 8-byte reads, contraction index
    // permuted like the transposing read), B = E via the transposing read
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
#pragma unroll
      for (int xs = 0; xs < DW / 32; ++xs) {
        struct { bf16x4 a, b; } t;
        t.a = *reinterpret_cast<const NHA_LDS bf16x4*>(Yt + (16 * rb + l16) * LDT + 32 * xs + 4 * kb);
        t.b = *reinterpret_cast<const NHA_LDS bf16x4*>(Yt + (16 * rb + l16) * LDT + 32 * xs + 16 + 4 * kb);
        const bf16x8 ya = __builtin_bit_cast(bf16x8, t);
        dsa[rb] = mfma16(ya, lds_frag_tr(Et, ELD, 32 * xs, 32 * xs + 16, 16 * wave, lane),
                         mfma16(ya, lds_frag_tr(El, ELD, 32 * xs, 32 * xs + 16, 16 * wave, lane), dsa[rb]));
      }
    }
    if (z + 1 == NZ) break;
    lds_barrier();   // (waits for this wave's reads)
    place(part);
    lds_barrier();
  }
  // through LDS to the thread that has the row's four slots
  constexpr int GLD = BT + 4;
  lfloat* const dl = (lfloat*)(NHA_LDS void*)Yt, * const gs = dl + BT * GLD;   // [64 r][GLD], [16 groups of rows][64]
  static_assert((BT * GLD + 16 * BT) * 4 <= (TILE + 2 * DW * ELD) * 2, "the rows of ds fit where the tiles were");
  lds_barrier();
#pragma unroll
  for (int rb = 0; rb < 4; ++rb)
#pragma unroll
    for (int q = 0; q < 4; ++q) dl[(16 * rb + 4 * kb + q) * GLD + col] = dsa[rb][q] * __expf(glast - grow[rb][q]);
  lds_barrier();
  f32x4 sum[4], run = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 3; q >= 0; --q) {
    const int r = 4 * rg + q;
    if (r >= vlo && r < R) {
      const f32x4 d = (f32x4){gi[q].x, gi[q].y, gi[q].z, gi[q].w} + *reinterpret_cast<const NHA_LDS f32x4*>(dl + r * GLD + gm);
      const f32x4 sv = {__uint_as_float(gsv[q].x << 16), __uint_as_float(gsv[q].x & 0xffff0000u), __uint_as_float(gsv[q].y << 16),
                        __uint_as_float(gsv[q].y & 0xffff0000u)};
      run += (f32x4){gx[q].x, gx[q].y, gx[q].z, gx[q].w} - sv * d;
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (__bf16)d[e];
      *reinterpret_cast<bf16x4*>(p.ds + (((int64_t)c0 + r - p.shift) * H + h) * BT + gm) = o;
    }
    sum[q] = run;   // over the later rows of the group
  }
  *reinterpret_cast<NHA_LDS f32x4*>(gs + rg * BT + gm) = run;
  lds_barrier();
  f32x4 later = {0.f, 0.f, 0.f, 0.f};
  for (int g = 15; g > rg; --g) later += *reinterpret_cast<const NHA_LDS f32x4*>(gs + g * BT + gm);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 4 * rg + q;
    if (r >= vlo && r < R) *reinterpret_cast<f32x4*>(p.dsi + (((int64_t)c0 + r) * H + h) * BT + gm) = sum[q] + later;
  }
  if (rg == 0) *reinterpret_cast<f32x4*>(p.gtot + ((int64_t)chunk * H + h) * BT + gm) = run + later;
}

template <int D, int TK>
int launch_dq(const WP& p, int NT, hipStream_t st) {
  const size_t lds = (size_t)4 * TK * (D + 16) * 2;
  static std::atomic<bool> configured{false};   // the attribute call is idempotent: a second thread may repeat it
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)bwd_dq_kernel<D, TK>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      set_error("nha_prefill_bwd: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
      return NHA_ERR_LAUNCH;
    }
    configured = true;
  }
  hipLaunchKernelGGL((bwd_dq_kernel<D, TK>), dim3(p.HQ, NT), dim3(256), lds, st, p);
  NHA_CHECK_LAUNCH("nha_prefill_bwd(window dq)");
  return NHA_OK;
}

template <int D, int TQ, bool SPLIT, int G>
int launch_dkv(const WP& p, int NT, hipStream_t st) {
  const size_t lds = (size_t)4 * TQ * (D + 16) * 2 + 4 * TQ * 4;
  static std::atomic<bool> configured{false};   // the attribute call is idempotent: a second thread may repeat it
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)bwd_dkv_kernel<D, TQ, SPLIT, G>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      set_error("nha_prefill_bwd: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
      return NHA_ERR_LAUNCH;
    }
    configured = true;
  }
  hipLaunchKernelGGL((bwd_dkv_kernel<D, TQ, SPLIT, G>), dim3(p.H, NT, SPLIT ? 2 : 1), dim3(256 * G), lds, st, p);
  NHA_CHECK_LAUNCH("nha_prefill_bwd(window dk, dv)");
  return NHA_OK;
}

WP make_wp(const NhaPrefillBwdArgs* a, const float* delta, const float* dvs) {
  WP p;
  p.ld = nullptr;
  p.q = (const bf16_t*)a->q_swa; p.k = (const bf16_t*)a->k_swa; p.v = (const bf16_t*)a->v;
  p.dout = (const bf16_t*)a->dout;
  p.lse_swa = a->lse_swa; p.lse_gsa = a->lse_gsa; p.delta = delta; p.dvs = dvs;
  p.dq = (bf16_t*)a->dq_swa; p.dk = (bf16_t*)a->dk_swa; p.dv = (bf16_t*)a->dv;
  p.cu = a->cu_seqlens; p.cidx = a->chunk_indices;
  p.HQ = a->HQ; p.H = a->H; p.NG = a->HQ / a->H; p.wl = a->wl; p.scale = a->scale;
  return p;
}

}  // namespace

bool bwd_window_mfma_supported(const NhaPrefillBwdArgs* a) {
  return a->dtype == NHA_DTYPE_BF16 && a->K == a->V && (a->K == 64 || a->K == 128 || a->K == 256) &&
         a->dlse_swa == nullptr && a->NT <= 65535;
}

int bwd_window_mfma_dq(const NhaPrefillBwdArgs* a, const float* delta, void* ld) {
  if (bwd_ring_supported(a)) return bwd_ring_dq(a, delta, (float2*)ld);
  if (bwd_ring256_dq_supported(a)) return bwd_ring256_dq(a, delta, (float2*)ld);
  WP p = make_wp(a, delta, nullptr);
  if (bwd_ring256_dkv_supported(a)) p.ld = (float2*)ld;
  hipStream_t st = (hipStream_t)a->stream;
  if (a->K == 64) return launch_dq<64, 64>(p, a->NT, st);
  if (a->K == 128) return launch_dq<128, 64>(p, a->NT, st);
  return launch_dq<256, 32>(p, a->NT, st);
}

int bwd_window_mfma_parts(const NhaPrefillBwdArgs* a) { return a->K == 256 ? bwd_ring256_dkv_parts(a) : bwd_ring_dkv_parts(a); }

int bwd_window_mfma_dkv(const NhaPrefillBwdArgs* a, const float* delta, const float* dvs, const void* ld, int parts, float* wk, float* wv) {
  if (bwd_ring_dkv_supported(a)) return bwd_ring_dkv(a, (const float2*)ld, dvs, parts, wk, wv);
  if (bwd_ring256_dkv_supported(a)) return bwd_ring256_dkv(a, (const float2*)ld, dvs, parts, wk, wv);
  const WP p = make_wp(a, delta, dvs);
  hipStream_t st = (hipStream_t)a->stream;
  // Eight waves per workgroup where all of them have a place at once: one workgroup per CU, at head size 64 two.  us, four / eight
  // waves: head size 64, 16 / 4 heads, W = 174, 63 to 624 workgroups 41 / 27, 49 / 39 (312), 61 / 61 (624), 16 / 16, W = 128, 15.7 /
  // 14.3 (480), 19 / 22 (752); 128, 8 / 2, W = 169 54 / 39 (240), 32 / 8, W = 571 114 / 79 (256), 4 / 4, W = 512 43 / 48 (512); 256, 8
  // / 2 48 / 38 (152), 86 / 98 (304).
  const bool two = (int64_t)a->H * a->NT * (a->K == 256 ? 2 : 1) <= (a->K == 64 ? 512 : 256);
  if (a->K == 64) return two ? launch_dkv<64, 64, false, 2>(p, a->NT, st) : launch_dkv<64, 64, false, 1>(p, a->NT, st);
  if (a->K == 128) return two ? launch_dkv<128, 64, false, 2>(p, a->NT, st) : launch_dkv<128, 64, false, 1>(p, a->NT, st);
  return two ? launch_dkv<256, 64, true, 2>(p, a->NT, st) : launch_dkv<256, 32, true, 1>(p, a->NT, st);
}

template <int D>
static int launch_slot_inter(const SP2& p, int NT, hipStream_t st) {
  constexpr int DWI = D > 128 ? 128 : D;   // columns per workgroup
  const size_t lds = (size_t)BT * (DWI + 16) * 2 + (size_t)2 * DWI * TLD * 2 + (size_t)2 * BT * TLD * 2;
  static std::atomic<bool> configured{false};   // the attribute call is idempotent: a second thread may repeat it
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)bwd_slot_inter_kernel<D, DWI>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      set_error("nha_prefill_bwd: cannot reserve LDS: %s", hipGetErrorString(e));
      return NHA_ERR_LAUNCH;
    }
    configured = true;
  }
  hipLaunchKernelGGL((bwd_slot_inter_kernel<D, DWI>), dim3(p.H, NT), dim3(256), lds, st, p);
  NHA_CHECK_LAUNCH("nha_prefill_bwd(slot branch, carried state gradient)");
  return NHA_OK;
}

int bwd_slot_inter(const NhaPrefillBwdArgs* a, const float* gc, const float* ek, const float* ev, const float* dks, float* dvs, const float* xg,
                   float* dsi, float* gtot) {
  SP2 p;
  p.kg = (const bf16_t*)a->k_gsa; p.v = (const bf16_t*)a->v; p.s = (const bf16_t*)a->s;
  p.gc = gc; p.ek = ek; p.ev = ev; p.dks = dks; p.dvs = dvs;
  p.xg = xg; p.dsi = dsi; p.gtot = gtot; p.ds = (bf16_t*)a->ds;
  p.dkg = (bf16_t*)a->dk_gsa;
  p.cu = a->cu_seqlens; p.cidx = a->chunk_indices;
  p.H = a->H; p.shift = a->shift;
  hipStream_t st = (hipStream_t)a->stream;
  if (a->K == 64) return launch_slot_inter<64>(p, a->NT, st);
  if (a->K == 128) return launch_slot_inter<128>(p, a->NT, st);
  return launch_slot_inter<256>(p, a->NT, st);
}

}  // namespace nha
