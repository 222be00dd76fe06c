// Exact recomputation of rows that an output pass of the matrix-core prefill cannot form (prefill_mfma.hip, prefill_ring.hip,
// prefill_ring256.hip): in fp32 vector arithmetic, row by row, from the same chunk-start states and gate table.
//
// An output pass writes the intra-chunk decay exp(gc_i - gc_j) as exp(gc_i - gr) * exp(gr - gc_j) with gr the gate cumsum at the
// start of j's 16-row sub-block, and caps the second exponent at DECAY_CLAMP.  Where a slot forgets faster than that (flags from the
// state pass), or where a row's window sums leave the range of their fixed softmax reference, the rows of the sub-block are formed
// again with the unfactored decay (<= 1): slot logits (nha_fla/ops/nha/chunk_fused.py:186-222), window logits, one softmax
// (:233-240), both reads (:242-283) and the branch LSEs (nha_fla/ops/nha/chunk.py:459-470).
//
// Who does it: the output pass at its end, in the workgroup that has formed the other rows.  A launch of its own (mfma_repair_kernel)
// takes 4 to 5 us of a call to find nothing to do -- three dependent misses: code, arguments, flags -- and 3 to 4 us of host time.
// The arguments are read again for it (arguments_again): kept from the beginning they cost ring_out_kernel 23 spilled scalar registers
// and 1.5 %.  Whole calls, the launch / inside, us: four heads of 128, 2 x 8192 tokens, W = 64 232.5 / 228.8, 2 x 16384, W = 2048 1170.5
// / 1170; head size 256, 32768 packed, W = 512 307 / 304, 4 x 8192, 8 / 2 heads, W = 2000 659 / 654; 16 heads of 128, 4 x 8192, W = 64
// 532 / 523.  At head size 64 with one or two heads the instance has room for it only at some cost: 16 heads, 2 x 8192, W = 2048 330 /
// 333, W = 64 176.6 / 172.7, 5003 tokens 74.4 / 72.4, 300 30.4 / 27.2; there short passes, EXACT_INSIDE_US as estimated from the rounds
// of workgroups, take it and the others the launch; so do two heads of 128 or 64 with more than a workgroup for every CU (no registers).  Every row flagged: four heads of 128, 4096 tokens, W = 512 23.5 / 22.7 ms, 4 heads
// of 256 7.3 / 7.1.
#pragma once
#include "mfma_common.h"

namespace nha {
namespace mf {

// Output passes of head size 64 up to this long form the exact rows themselves.
constexpr double EXACT_INSIDE_US = 100;
// units of 32 keys that a workgroup walks on average, from the call's totals
inline double window_units(const MP& p) {
  const double len = (double)p.T_tot / p.N, w = p.wl < 0 || p.wl > len / 2 ? len / 2 : p.wl;
  return (w + BT) / 32;
}

// Floats of LDS: the states and gates of a chunk, and what each group of 256 threads keeps of its row.  HV: the v-state too, where
// there is room for it.
template <int D, int GROUPS, bool HV>
struct ExactSmem {
  static constexpr int LDH = D + 1;
  static constexpr int SHARED = MS * LDH + (HV ? MS * D : 0) + BT * MS;
  static constexpr int ROW = 2 * D + 2 * MS + 2 * BT + 256 + 4 + BT;
  static constexpr size_t bytes = (size_t)(SHARED + GROUPS * ROW) * 4;
};

// max and sum over a group of 256 threads (red: 4 floats of the group), all groups of the workgroup at once
__device__ __forceinline__ float group_max(float v, float* red, int t) {
  v = wave_max(v);
  __syncthreads();
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
__device__ __forceinline__ float group_sum(float v, float* red, int t) {
  v = wave_sum(v);
  __syncthreads();
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// The rows of the 16-row blocks in `bits` of a chunk (rows c0 .. of the sequence [bos, eos)) for the query heads hq0 .. hq0 + nheads - 1
// of kv-head h.  GROUPS groups of 256 threads take a head each, or rows of the one head there is; whoever has none left repeats the
// last one.  Called by the whole workgroup; rsm: ExactSmem<D, GROUPS, HV>::bytes that nobody uses any more.
template <int D, int GROUPS, bool HV = true>
__device__ __forceinline__ void exact_rows(const MP& p, float* rsm, int chunk, int h, int hq0, int nheads, int bits) {
  typedef ExactSmem<D, GROUPS, HV> S;
  constexpr int LDH = S::LDH, NT = 256 * GROUPS;
  const int tid = threadIdx.x, t = tid & 255, group = GROUPS > 1 ? tid >> 8 : 0;
  float* const hk = rsm;                     // [MS][LDH] true chunk-start k-state, transposed
  float* const hv = hk + MS * LDH;           // [MS][D]   true chunk-start v-state
  float* const gcl = hv + (HV ? MS * D : 0); // [BT][MS]  gate cumsum
  float* const qg = rsm + S::SHARED + group * S::ROW;   // [D] scaled slot-branch query
  float* const qs = qg + D;                  // [D] scaled window query
  float* const okl = qs + D;                 // [MS] slot logits -> probabilities
  float* const gct = okl + MS;               // [MS] gate cumsum of the row
  float* const Aj = gct + MS;                // [BT]
  float* const Avj = Aj + BT;                // [BT]
  float* const pw = Avj + BT;                // [256]
  float* const red = pw + 256;               // [4]
  int* const src = (int*)(red + 4);          // [BT]
  const int H = p.H, HQ = p.HQ;
  const int64_t cg = (int64_t)chunk * H + h;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int c0 = bos + it * BT;
  const int rows = (eos - c0) < BT ? (eos - c0) : BT;
  for (int e = tid; e < MS * D; e += NT) {
    const int m = e / D, d = e % D;
    hk[m * LDH + d] = bf16_to_f32(p.hkT[(cg * MS + m) * D + d]);
    if (HV) hv[m * D + d] = bf16_to_f32(p.hvc[(cg * MS + m) * D + d]);
  }
  for (int e = tid; e < BT * MS; e += NT) gcl[e] = p.gc[cg * BT * MS + e];

  auto first_key = [&](int x) { return p.wl < 0 ? bos : (x - p.wl > bos ? x - p.wl : bos); };
  const bool by_row = nheads == 1;
  for (int a = 0; a < nheads; a += GROUPS)
  for (int r0 = 0; r0 < rows; r0 += by_row ? GROUPS : 1) {
    if (!((bits >> (r0 >> 4)) & 1)) continue;
    const int hq = hq0 + (a + group < nheads ? a + group : nheads - 1);
    const int rx = by_row ? r0 + GROUPS - 1 : r0, rlast = rx < rows ? rx : rows - 1;   // the last row that a group takes
    const int r = by_row && r0 + group < rlast ? r0 + group : rlast;
    const int tok = c0 + r;
    __syncthreads();   // state tables are in place; the previous row is finished
    const bf16_t* qsw = p.q_swa + ((int64_t)tok * HQ + hq) * D;
    const bf16_t* qgs = p.q_gsa + ((int64_t)tok * HQ + hq) * D;
    for (int i = t; i < D; i += 256) {
      qg[i] = bf16_to_f32(qgs[i]) * p.scale;
      qs[i] = bf16_to_f32(qsw[i]) * p.scale;
    }
    if (t < MS) gct[t] = gcl[r * MS + t];
    if (t < BT) {
      const int tl = it * BT + t - p.shift;
      src[t] = (t <= r && tl >= 0) ? bos + tl : -1;
    }
    __syncthreads();
    if (t < BT) {
      const int sj = src[t];
      Aj[t] = sj >= 0 ? dot_row<bf16_t>(qg, p.k_gsa + ((int64_t)sj * H + h) * D, D) : 0.f;
    }
    __syncthreads();
    float lmax = -INFINITY;
    if (t < MS) {
      const int m = t;
      float acc = 0.f;
      for (int d = 0; d < D; ++d) acc += qg[d] * hk[m * LDH + d];
      acc *= expf(gct[m]);
      for (int j = 0; j <= r; ++j) {
        const int sj = src[j];
        if (sj >= 0) acc += Aj[j] * bf16_to_f32(p.s[((int64_t)sj * H + h) * MS + m]) * expf(gct[m] - gcl[j * MS + m]);
      }
      okl[m] = acc;
      lmax = acc;
    }
    const float mg = group_max(lmax, red, t);
    const float lg = group_sum(t < MS ? expf(okl[t] - mg) : 0.f, red, t);
    const int lo = first_key(tok);
    float wm = -INFINITY, wsum = 0.f;
    for (int j = lo + t; j <= tok; j += 256) {
      const float d = dot_row<bf16_t>(qs, p.k_swa + ((int64_t)j * H + h) * D, D);
      if (d > wm) {
        wsum = wsum * expf(wm - d) + 1.f;
        wm = d;
      } else {
        wsum += expf(d - wm);
      }
    }
    const float mw = group_max(wm, red, t);
    const float lw = group_sum(wm == -INFINITY ? 0.f : wsum * expf(wm - mw), red, t);
    if (t == 0) {
      if (p.lse_gsa) p.lse_gsa[(int64_t)tok * HQ + hq] = mg + logf(lg);
      if (p.lse_swa) p.lse_swa[(int64_t)tok * HQ + hq] = mw + logf(lw);
    }
    const float mt = fmaxf(mg, mw);
    const float inv = 1.f / (lg * expf(mg - mt) + lw * expf(mw - mt));
    __syncthreads();
    if (t < MS) okl[t] = expf(okl[t] - mt) * inv;
    __syncthreads();
    if (t < BT) {
      const int sj = src[t];
      float acc = 0.f;
      if (sj >= 0) {
        const bf16_t* srow = p.s + ((int64_t)sj * H + h) * MS;
        for (int m = 0; m < MS; ++m) acc += okl[m] * bf16_to_f32(srow[m]) * expf(gct[m] - gcl[t * MS + m]);
      }
      Avj[t] = acc;
    }
    __syncthreads();
    float acc = 0.f;   // value column t (D <= 256 == threads of a group)
    if (t < D) {
      for (int m = 0; m < MS; ++m) acc += okl[m] * expf(gct[m]) * (HV ? hv[m * D + t] : bf16_to_f32(p.hvc[(cg * MS + m) * D + t]));
      for (int j = 0; j <= r; ++j) {
        const int sj = src[j];
        if (sj >= 0) acc += Avj[j] * bf16_to_f32(p.v[((int64_t)sj * H + h) * D + t]);
      }
    }
    for (int jb = lo; jb - lo <= c0 + rlast - first_key(c0 + r0); jb += 256) {   // as often in every group
      const int j = jb + t;
      __syncthreads();
      pw[t] = j <= tok ? expf(dot_row<bf16_t>(qs, p.k_swa + ((int64_t)j * H + h) * D, D) - mt) * inv : 0.f;
      __syncthreads();
      const int cnt = (tok - jb + 1) < 256 ? (tok - jb + 1) : 256;
      if (t < D)
        for (int x = 0; x < cnt; ++x) acc += pw[x] * bf16_to_f32(p.v[((int64_t)(jb + x) * H + h) * D + t]);
    }
    if (t < D) p.o[((int64_t)tok * HQ + hq) * D + t] = f32_to_bf16(acc);
  }
}

// The kernel's arguments (its only parameter), read anew: what a rare branch at the end of a kernel takes of them would otherwise be
// kept from the beginning, in scalar registers that the loop before it does not have to spare.
__device__ __forceinline__ const MP& arguments_again() {
  const __attribute__((address_space(4))) void* a = (const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return *(const MP*)a;
}

// This wave's stores have been written and everybody's LDS reads are done: exact_rows may write over both.
__device__ __forceinline__ void before_exact() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();
}

}  // namespace mf
}  // namespace nha
