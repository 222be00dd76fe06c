// Decode step for few (sequence, kv-head) pairs on gfx950: the work of one pair spread over several workgroups.
// Same calls as decode_mfma.hip (bf16, K == V == D in {64,128,256}, M == 64 slots, up to 8 query heads per kv-head,
// window or ring mode, pre-rotated query or, up to head size 128, cos / sin tables).
//
// A pair's step is cut into tasks of one WAVE that need nothing from each other:
//   slot task    8 of the 64 slots: their columns of the k-state and rows of the v-state are updated
//                (nha_fla/ops/nha/fused_recurrent.py:305, :342-349), their logits, their softmax weights relative to
//                the task's own maximum, and their part of the slot read (:416);
//   window task  32 keys of the window: S^T = K Q^T and O^T += V^T P^T on the matrix cores as in decode_mfma.hip.
// P workgroups of four waves share a pair's tasks; every wave leaves (max, sum, O) of what it did in LDS, a workgroup
// merges its waves, and the workgroup of the pair that arrives last (a counter in the caller's scratch) merges the
// workgroups' partials under one softmax, writes the output and puts the new token into the ring.  The new token goes
// into the ring there and not earlier because its row is the popped entry's, which every slot task reads.
#include "decode_common.h"

namespace nha {
namespace {

using namespace dec;

constexpr int NW = 4;          // waves per workgroup
constexpr int ST = 8;          // slots per slot task
constexpr int NST = MS / ST;   // slot tasks of a pair
constexpr int CUS = 256;       // compute units
constexpr int MAX_SPLIT = CUS / 2;   // pairs of a call that are still split (split_of)

template <int D, int G> struct Lds {
  static constexpr int LDT = D + 16;               // bf16 row stride of a V tile
  static constexpr int TILE = 32 * LDT / 2;        // floats of a wave's V tile, later its window partial [G][D]
  static constexpr int OS = NW * TILE;             // [NW][G][D] slot partials
  static constexpr int P = OS + NW * G * D;        // [NW][G][ST] slot weights of the running task
  static constexpr int AL = P + NW * G * ST;       // [NW][G] rescale of what the wave has summed so far
  static constexpr int ML = AL + NW * G;           // [2 NW][2][G] (max, sum) of every partial: slots, then windows
  static constexpr int FLAG = ML + 4 * NW * G;     // last-arriver flag
  static constexpr size_t BYTES = (FLAG + 4) * sizeof(float);
  static_assert(TILE >= G * D, "a wave's window partial fits its V tile");
};

// CPL consecutive bf16 as floats (CPL = 1, 2, 4: 2, 4 or 8 bytes)
template <int CPL>
__device__ __forceinline__ void ld_bf(const bf16_t* p, float* o) {
  if constexpr (CPL == 1) {
    o[0] = bf16_to_f32(p[0]);
  } else if constexpr (CPL == 2) {
    const uint32_t x = *reinterpret_cast<const uint32_t*>(p);
    o[0] = __uint_as_float(x << 16); o[1] = __uint_as_float(x & 0xffff0000u);
  } else {
    const uint2 x = *reinterpret_cast<const uint2*>(p);
    o[0] = __uint_as_float(x.x << 16); o[1] = __uint_as_float(x.x & 0xffff0000u);
    o[2] = __uint_as_float(x.y << 16); o[3] = __uint_as_float(x.y & 0xffff0000u);
  }
}
template <int CPL>
__device__ __forceinline__ void ld_f(const float* p, float* o) {
  if constexpr (CPL == 1) {
    o[0] = p[0];
  } else if constexpr (CPL == 2) {
    const float2 x = *reinterpret_cast<const float2*>(p);
    o[0] = x.x; o[1] = x.y;
  } else {
    const float4 x = *reinterpret_cast<const float4*>(p);
    o[0] = x.x; o[1] = x.y; o[2] = x.z; o[3] = x.w;
  }
}
template <int CPL>
__device__ __forceinline__ void st_f(float* p, const float* v) {
  if constexpr (CPL == 1) p[0] = v[0];
  else if constexpr (CPL == 2) *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
  else *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}

// The partner of a lane across bit MASK.  Within 16 lanes these are DPP moves (no LDS round trip); 4 and 8 mirror the
// lower bits as well, which a caller whose values agree over them, or who sums over them next, does not notice.
template <int MASK>
__device__ __forceinline__ float across(float v) {
  const int x = __float_as_int(v);
  constexpr int ctrl = MASK == 1 ? 0xB1 : MASK == 2 ? 0x4E : MASK == 4 ? 0x141 : 0x140;   // quad_perm, row_half_mirror, row_mirror
  if constexpr (MASK <= 8) return __int_as_float(__builtin_amdgcn_update_dpp(x, x, ctrl, 0xf, 0xf, true));
  else return __shfl_xor(v, MASK, 64);
}

// Sum over the wave of N values per lane (N a power of two up to 64): afterwards lane l holds the sum of value
// l >> (6 - log2 N).  Halving exchange: a step sends half of what is left, 63 exchanges for 64 values where summing
// each value over the wave takes 384.
template <int N, int MASK>
__device__ __forceinline__ float wave_scatter_sum(float* v, int lane) {
  if constexpr (MASK == 0) {
    return v[0];
  } else if constexpr (N == 1) {
    v[0] += across<MASK>(v[0]);
    return wave_scatter_sum<1, MASK / 2>(v, lane);
  } else {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      if constexpr (MASK == 32) {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + N / 2]), false, false);
        v[i] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
      } else if constexpr (MASK == 16) {
        const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + N / 2]), false, false);
        v[i] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
      } else {
        const float keep = (lane & MASK) ? v[i + N / 2] : v[i];
        const float send = (lane & MASK) ? v[i] : v[i + N / 2];
        v[i] = keep + across<MASK>(send);
      }
    }
    return wave_scatter_sum<N / 2, MASK / 2>(v, lane);
  }
}

// Stores and loads at device scope: they go past the L2 of an XCD, so what one workgroup stores and waits for
// (s_waitcnt vmcnt) the workgroups of other XCDs read without either side writing back or invalidating a cache.  A
// release fence instead writes the whole L2 back for every workgroup, one after the other: 64 pairs of 4 workgroups took
// 35 us with it, 14 us without the split.
__device__ __forceinline__ void st_agent(float* p, float x, float y) {
  const uint64_t v = (uint64_t)__float_as_uint(y) << 32 | __float_as_uint(x);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 ld_agent(const float* p) {
  const uint64_t v = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}

constexpr int log2c(int x) { return x <= 1 ? 0 : 1 + log2c(x / 2); }

// scratch: [MAX_SPLIT] counters (zero before the first step and after every step, and in the same place for every call, so
// that calls of other sizes may share the scratch), then the workgroups' partials
// [pairs][P][G][D] and their [pairs][P][G] (max, sum)
struct SplitArgs {
  NhaDecodeArgs a;
  int P;
  int* counter;
  float* po;
  float* pml;
};

template <int D, int G, bool ROT>
__global__ __launch_bounds__(64 * NW, 2) void decode_split_kernel(const SplitArgs sa) {
  typedef Lds<D, G> L;
  constexpr int LDT = L::LDT;
  constexpr int KS = D / 32;    // MFMA k-steps over the head dim
  constexpr int NVT = D / 16;   // 16-row blocks of O^T == 16-byte V loads per lane and block
  constexpr int LV = D / 8;     // lanes per V row
  constexpr int RV = 64 / LV;   // rows per wave-wide load
  constexpr int CPL = D / 64;   // k-state rows / v-state columns of a lane
  constexpr int M = MS;
  extern __shared__ __align__(16) float lds_raw[];
  const NhaDecodeArgs& a = sa.a;
  const int W = a.W, H = a.H, HQ = a.HQ, NG = HQ / H, P = sa.P;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, qd = lane >> 4;

  // Workgroups are dealt to the 8 XCDs in launch order: the workgroups of one pair sit 8 apart and so on one XCD,
  // where they find the state lines they share (a slot task takes 32 bytes of each k-state row) and each other's
  // partials in one L2.  What is left over of a multiple of 8 pairs is dealt pair by pair.
  int bh, p;
  {
    const int pairs = a.B * H, full = pairs & ~7, L0 = blockIdx.x;
    if (L0 < full * P) {
      const int j = L0 >> 3;
      bh = (j / P) * 8 + (L0 & 7);
      p = j % P;
    } else {
      const int rest = pairs - full, j = L0 - full * P;
      bh = full + j % rest;
      p = j / rest;
    }
  }
  const int b = bh / H, h = bh % H;
  const float qscale = a.scale * LOG2E;
  const int S = P * NW, ws = p * NW + wave;   // wave slots of the pair

  const bool ring = a.mode == NHA_DECODE_RING;
  int slot = -1, nvalid = W, cnt = 0;
  if (ring) {
    cnt = a.count[b];
    slot = cnt % W;
    nvalid = cnt + 1 < W ? cnt + 1 : W;
    if (a.count_next && h == 0 && p == 0 && tid == 0) a.count_next[b] = cnt + 1;
  }

  float* const os = lds_raw + L::OS + wave * G * D;
  float* const pw = lds_raw + L::P + wave * G * ST;
  float* const al = lds_raw + L::AL + wave * G;
  float* const ml = lds_raw + L::ML;

  // ================= slot tasks ws, ws + S, ... ====================================================
  constexpr int N = G * ST, SH = 6 - log2c(N);   // lane l holds logit l >> SH of the task: head, then slot
  float mrun = -INFINITY, lrun = 0.f;            // of this lane's head
  if (ws < NST) {
    float O[G][CPL];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int c = 0; c < CPL; ++c) O[g][c] = 0.f;
    for (int t = ws; t < NST; t += S) {
      const int s0 = t * ST;
      // every load of the task up front: states and queries first (they do not depend on the counter), then the
      // popped entry
      float hk[CPL][ST], hv[ST][CPL], q[G][CPL];
      const int64_t kbase = ((int64_t)bh * D + CPL * lane) * M + s0, vbase = ((int64_t)bh * M + s0) * D + CPL * lane;
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        if (a.hk_in) {
          Elem<float>::ld8(a.hk_in + kbase + c * M, hk[c]);
        } else {
#pragma unroll
          for (int s = 0; s < ST; ++s) hk[c][s] = 0.f;
        }
      }
#pragma unroll
      for (int s = 0; s < ST; ++s) {
        if (a.hv_in) {
          ld_f<CPL>(a.hv_in + vbase + s * D, hv[s]);
        } else {
#pragma unroll
          for (int c = 0; c < CPL; ++c) hv[s][c] = 0.f;
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int gq = g < NG ? g : NG - 1;
        ld_bf<CPL>((const bf16_t*)a.q + ((int64_t)b * HQ + h * NG + gq) * D + CPL * lane, q[g]);
      }
      bool has_pop = true;
      const bf16_t *kpop, *vpop, *gpop, *spop = nullptr;
      if (ring) {
        has_pop = cnt >= W;
        const int64_t row = ((int64_t)b * W + slot) * H + h;
        kpop = (const bf16_t*)a.ring_kg + row * D;
        vpop = (const bf16_t*)a.ring_v + row * D;
        gpop = (const bf16_t*)a.ring_g + row * M;
      } else {
        kpop = (const bf16_t*)a.k_pop + (int64_t)bh * D;
        vpop = (const bf16_t*)a.v_pop + (int64_t)bh * D;
        gpop = (const bf16_t*)a.g_pop + (int64_t)bh * M;
        if (a.s_pop) spop = (const bf16_t*)a.s_pop + (int64_t)bh * M;
      }
      float kp[CPL], vp[CPL], eg[ST], sg[ST];
      ld_bf<CPL>(kpop + CPL * lane, kp);
      ld_bf<CPL>(vpop + CPL * lane, vp);
      Elem<bf16_t>::ld8(gpop + s0, eg);
      if (spop) Elem<bf16_t>::ld8(spop + s0, sg);
#pragma unroll
      for (int s = 0; s < ST; ++s) {
        const float e = expf(eg[s]);
        eg[s] = has_pop ? e : 1.f;
        sg[s] = has_pop ? (spop ? sg[s] : 1.f - e) : 0.f;
      }
      // a ring that is not full pops nothing: its row holds no token yet and may hold anything, NaN included, which a zero
      // strength would not keep out
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        kp[c] = has_pop ? kp[c] : 0.f;
        vp[c] = has_pop ? vp[c] : 0.f;
      }
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
#pragma unroll
        for (int s = 0; s < ST; ++s) hk[c][s] = hk[c][s] * eg[s] + kp[c] * sg[s];
        if (a.hk_out) Elem<float>::st8(a.hk_out + kbase + c * M, hk[c]);
      }
      float acc[N];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int s = 0; s < ST; ++s) {
          float x = 0.f;
#pragma unroll
          for (int c = 0; c < CPL; ++c) x += q[g][c] * hk[c][s];
          acc[g * ST + s] = x;
        }
      const float v = wave_scatter_sum<N, 32>(acc, lane) * qscale;
      float mx = v;
      mx = fmaxf(mx, across<1 << SH>(mx));
      mx = fmaxf(mx, across<2 << SH>(mx));
      mx = fmaxf(mx, across<4 << SH>(mx));
      const float mnew = fmaxf(mrun, mx), ref = mnew == -INFINITY ? 0.f : mnew;   // eight slots may all weigh nothing
      const float alpha = fexp2(mrun - ref), e = fexp2(v - ref);
      float sum = e;
      sum += across<1 << SH>(sum);
      sum += across<2 << SH>(sum);
      sum += across<4 << SH>(sum);
      lrun = lrun * alpha + sum;
      mrun = mnew;
      pw[lane >> SH] = e;
      al[lane >> (SH + 3)] = alpha;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's own area: no barrier
#pragma unroll
      for (int s = 0; s < ST; ++s) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) hv[s][c] = hv[s][c] * eg[s] + sg[s] * vp[c];
        if (a.hv_out) st_f<CPL>(a.hv_out + vbase + s * D, hv[s]);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float r = al[g];
        float pr[ST];
        Elem<float>::ld8(pw + g * ST, pr);
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          float x = O[g][c] * r;
#pragma unroll
          for (int s = 0; s < ST; ++s) x += pr[s] * hv[s][c];
          O[g][c] = x;
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int g = 0; g < G; ++g) st_f<CPL>(os + g * D + CPL * lane, O[g]);
    if (lrun != lrun) mrun = INFINITY;   // a maximum does not carry NaN: without this the merge would pass the part over
  }
  ml[(2 * wave) * G + (lane >> (SH + 3))] = mrun;      // -inf and 0 where the wave had no slot task
  ml[(2 * wave + 1) * G + (lane >> (SH + 3))] = lrun;

  // ================= window tasks: blocks S-1-ws, +S, ... (the waves without slot tasks first) =======
  lbf16* X = (lbf16*)(NHA_LDS void*)(lds_raw + wave * L::TILE);
  const int nblk = (nvalid + 31) >> 5;
  float wmax = -INFINITY, wsum = 0.f;
  const int blk0 = S - 1 - ws;
  if (blk0 < nblk) {
    const bf16_t* kwin = (const bf16_t*)(ring ? a.ring_k : a.win_k) + ((int64_t)b * W * H + h) * D;
    const bf16_t* vwin = (const bf16_t*)(ring ? a.ring_v : a.win_v) + ((int64_t)b * W * H + h) * D;
    const bf16_t* knew = ring ? (const bf16_t*)a.k_new + (int64_t)bh * D : nullptr;
    const bf16_t* vnew = ring ? (const bf16_t*)a.v_new + (int64_t)bh * D : nullptr;
    const bf16_t* ctab = ROT ? (const bf16_t*)a.cos + (int64_t)b * a.cos_sb : nullptr;
    const bf16_t* stab = ROT ? (const bf16_t*)a.sin + (int64_t)b * a.cos_sb : nullptr;
    const uint32_t rstride = (uint32_t)H * D;
    // rows past the valid range are clamped to the last valid row (finite data); their logits are masked below.
    // Ring row `slot` is the new token, read from k_new / v_new.
    auto load_block = [&](uint4(&kr)[2 * KS], uint4(&vr)[NVT], int blk) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        int w = 32 * blk + 16 * t + l16;
        w = w < nvalid ? w : nvalid - 1;
        const bf16_t* pr = kwin + (uint32_t)w * rstride;
        const bf16_t* row = (w == slot ? knew : pr) + 8 * qd;
#pragma unroll
        for (int j = 0; j < KS; ++j) kr[t * KS + j] = ld16_stream(row + 32 * j);
      }
#pragma unroll
      for (int u = 0; u < NVT; ++u) {
        int w = 32 * blk + u * RV + lane / LV;
        w = w < nvalid ? w : nvalid - 1;
        const bf16_t* pr = vwin + (uint32_t)w * rstride;
        const bf16_t* row = (w == slot ? vnew : pr) + 8 * (lane % LV);
        vr[u] = ld16_stream(row);
      }
    };
    uint4 kr[2 * KS], vr[NVT];
    uint4 cr[ROT ? 2 * KS : 1], sr[ROT ? 2 * KS : 1];   // cos / sin pieces of the block's keys
    auto load_tables = [&](int blk) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        int w = 32 * blk + 16 * t + l16;
        w = w < nvalid ? w : nvalid - 1;
        const int64_t off = (int64_t)w * a.cos_sw + 8 * qd;
#pragma unroll
        for (int j = 0; j < KS; ++j) {
          cr[ROT ? t * KS + j : 0] = *reinterpret_cast<const uint4*>(ctab + off + 32 * j);
          sr[ROT ? t * KS + j : 0] = *reinterpret_cast<const uint4*>(stab + off + 32 * j);
        }
      }
    };
    load_block(kr, vr, blk0);
    if constexpr (ROT) load_tables(blk0);
    // window-query B fragments: lane (head l%16, piece l/16) of each 32-wide k-step
    bf16x8 qf[KS];
    {
      uint4 qx[KS];
      const bf16_t* qsrc = ROT ? (const bf16_t*)a.q : (const bf16_t*)a.sq;
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        qx[j] = make_uint4(0, 0, 0, 0);
        if (l16 < NG) qx[j] = *reinterpret_cast<const uint4*>(qsrc + ((int64_t)b * HQ + h * NG + l16) * D + 32 * j + 8 * qd);
      }
      if constexpr (ROT) {   // the query's own position is the last row of the tables
        const bf16_t* cq = ctab + (int64_t)(W - 1) * a.cos_sw + 8 * qd;
        const bf16_t* sq_ = stab + (int64_t)(W - 1) * a.cos_sw + 8 * qd;
#pragma unroll
        for (int j = 0; j < KS / 2; ++j) {
          const uint4 ca = *reinterpret_cast<const uint4*>(cq + 32 * j), sa_ = *reinterpret_cast<const uint4*>(sq_ + 32 * j);
          const uint4 cb = *reinterpret_cast<const uint4*>(cq + 32 * (j + KS / 2)), sb = *reinterpret_cast<const uint4*>(sq_ + 32 * (j + KS / 2));
          rope8(qx[j], qx[j + KS / 2], ca, sa_, cb, sb);
        }
      }
#pragma unroll
      for (int j = 0; j < KS; ++j) qf[j] = as_bf16x8(qx[j]);
    }
    f32x4 O[NVT];
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt) O[vt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int blk = blk0; blk < nblk; blk += S) {
      if constexpr (ROT) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int j = 0; j < KS / 2; ++j) {
            const int x = t * KS + j, y = x + KS / 2;
            rope8(kr[x], kr[y], cr[x], sr[x], cr[y], sr[y]);
          }
      }
      f32x4 S0 = {0.f, 0.f, 0.f, 0.f}, S1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < KS; ++j) S0 = mfma16(as_bf16x8(kr[j]), qf[j], S0);
#pragma unroll
      for (int j = 0; j < KS; ++j) S1 = mfma16(as_bf16x8(kr[KS + j]), qf[j], S1);
#pragma unroll
      for (int u = 0; u < NVT; ++u) {
        const u32x4 x = {vr[u].x, vr[u].y, vr[u].z, vr[u].w};
        *reinterpret_cast<NHA_LDS u32x4*>(X + (u * RV + lane / LV) * LDT + 8 * (lane % LV)) = x;
      }
      __builtin_amdgcn_sched_barrier(0);
      if (blk + S < nblk) {   // wave-uniform: the next block's loads fly during this block's softmax and products
        load_block(kr, vr, blk + S);
        if constexpr (ROT) load_tables(blk + S);
      }
      __builtin_amdgcn_sched_barrier(0);
      // S^T rows of this lane: keys 32*blk + 4*qd + r (S0) and + 16 (S1), head l16
      const int wb = 32 * blk + 4 * qd;
      float s[8];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[r] = wb + r < nvalid ? S0[r] * qscale : -INFINITY;
        s[4 + r] = wb + 16 + r < nvalid ? S1[r] * qscale : -INFINITY;
      }
      float mx = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
      mx = max_over_rows(mx);
      const float mnew = fmaxf(wmax, mx);
      const float alpha = fexp2(wmax - mnew);
      wmax = mnew;
      float ps = 0.f;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        s[r] = fexp2(s[r] - mnew);
        ps += s[r];
      }
      wsum = wsum * alpha + ps;
      bf16x8 Pf;
#pragma unroll
      for (int r = 0; r < 8; ++r) Pf[r] = (__bf16)s[r];
#pragma unroll
      for (int vt = 0; vt < NVT; ++vt) {
        O[vt] *= alpha;
        O[vt] = mfma16(lds_frag_tr(X, LDT, 16 * vt, lane), Pf, O[vt]);
      }
    }
    wsum = sum_over_rows(wsum);
    if (wsum != wsum) wmax = INFINITY;   // as for the slots: the merge gives NaN
    // O^T[v = 16*vt + 4*qd + r][head l16] -> wave-private fp32 [G][D] over this wave's V tile
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    lfloat* Ow = (lfloat*)(NHA_LDS void*)X;
    if (l16 < G) {
#pragma unroll
      for (int vt = 0; vt < NVT; ++vt) *reinterpret_cast<NHA_LDS f32x4*>(Ow + l16 * D + 16 * vt + 4 * qd) = O[vt];
    }
  }
  if (qd == 0 && l16 < G) {
    ml[(2 * (NW + wave)) * G + l16] = wmax;
    ml[(2 * (NW + wave) + 1) * G + l16] = wsum;
  }
  lds_barrier();

  // ================= the workgroup's partial: its waves' slot and window parts under one maximum =====
  // four consecutive columns of one head per thread
  constexpr int NT = 64 * NW;
  auto store_out = [&](int i, const f32x4& num, float den) {
    const int g = i / D;
    if (g >= NG) return;
    const float r = 1.f / den;
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (__bf16)(num[e] * r);
    *reinterpret_cast<bf16x4*>((bf16_t*)a.o + ((int64_t)b * HQ + h * NG) * D + i) = o;
  };
  for (int i = 4 * tid; i < G * D; i += 4 * NT) {
    const int g = i / D;
    float mt = -INFINITY, mx[2 * NW];
#pragma unroll
    for (int x = 0; x < 2 * NW; ++x) mt = fmaxf(mt, mx[x] = ml[2 * x * G + g]);
    f32x4 num = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
#pragma unroll
    for (int x = 0; x < 2 * NW; ++x) {
      if (mx[x] != -INFINITY) {   // the same for a whole wave: the columns of a head
        const float c = fexp2(mx[x] - mt);
        const float* src = lds_raw + (x < NW ? L::OS + x * G * D : (x - NW) * L::TILE) + i;
        num += *reinterpret_cast<const f32x4*>(src) * c;
        den += ml[(2 * x + 1) * G + g] * c;
      }
    }
    if (P == 1) {
      store_out(i, num, den);
    } else {
      const int64_t part = (int64_t)bh * P + p;
      st_agent(sa.po + part * (G * D) + i, num[0], num[1]);
      st_agent(sa.po + part * (G * D) + i + 2, num[2], num[3]);
      if (i == g * D) st_agent(sa.pml + (part * G + g) * 2, mt, den);
    }
  }
  if (P > 1) {
    int* flag = (int*)(lds_raw + L::FLAG);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's partials have reached the device's coherence point
    __syncthreads();
    if (tid == 0) {
      const int arrived = __hip_atomic_fetch_add(sa.counter + bh, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = arrived == P - 1;
      if (arrived == P - 1) __hip_atomic_store(sa.counter + bh, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*flag) return;
    for (int i = 4 * tid; i < G * D; i += 4 * NT) {
      const int g = i / D;
      const float* pm = sa.pml + ((int64_t)bh * P * G + g) * 2;
      const float* po = sa.po + (int64_t)bh * P * (G * D) + i;
      float mt = -INFINITY, den = 0.f;
      f32x4 num = {0.f, 0.f, 0.f, 0.f};
      for (int x0 = 0; x0 < P; x0 += 4) {   // four workgroups' partials are requested together
        float2 m[4], lo[4], hi[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int x = x0 + u < P ? x0 + u : P - 1;
          m[u] = ld_agent(pm + x * (2 * G));
          lo[u] = ld_agent(po + (int64_t)x * (G * D));
          hi[u] = ld_agent(po + (int64_t)x * (G * D) + 2);
        }
        float mn = mt;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (x0 + u >= P) m[u].x = -INFINITY;
          mn = fmaxf(mn, m[u].x);
        }
        if (mn == -INFINITY) continue;
        const float r = fexp2(mt - mn);
        num *= r;
        den *= r;
        mt = mn;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float c = fexp2(m[u].x - mt);   // 0 for a workgroup that found no task: max -inf
          num += (f32x4){lo[u].x, lo[u].y, hi[u].x, hi[u].y} * c;
          den += m[u].y * c;
        }
      }
      store_out(i, num, den);
    }
  }
  if (ring) {
    // every task of the pair has read the popped entry: the new token takes its ring slot
    const int64_t row = ((int64_t)b * W + slot) * H + h;
    const int x = tid & 63;
    if (wave == 0 && x < D / 8)
      reinterpret_cast<uint4*>((bf16_t*)a.ring_k + row * D)[x] = reinterpret_cast<const uint4*>((const bf16_t*)a.k_new + (int64_t)bh * D)[x];
    if (wave == 1 && x < D / 8)
      reinterpret_cast<uint4*>((bf16_t*)a.ring_kg + row * D)[x] = reinterpret_cast<const uint4*>((const bf16_t*)a.kg_new + (int64_t)bh * D)[x];
    if (wave == 2 && x < D / 8)
      reinterpret_cast<uint4*>((bf16_t*)a.ring_v + row * D)[x] = reinterpret_cast<const uint4*>((const bf16_t*)a.v_new + (int64_t)bh * D)[x];
    if (wave == 3 && x < M / 8)
      reinterpret_cast<uint4*>((bf16_t*)a.ring_g + row * M)[x] = reinterpret_cast<const uint4*>((const bf16_t*)a.g_new + (int64_t)bh * M)[x];
  }
}

int group_of(const NhaDecodeArgs* a) {
  int G = 1;
  while (G < a->HQ / a->H) G <<= 1;
  return G;
}

// Workgroups per pair; 0: the call keeps decode_mfma_kernel.  us per step (graph of 20 steps) without / with the split:
//   pairs   G  D     W = 64        W = 256       W = 2048
//      4    8  128   16.6 /  7.3   18.0 /  7.4   40.5 /  9.7
//     24    4  128   12.1 /  6.9   14.2 /  7.2   41.3 / 12.7
//     64    4  128   12.6 /  7.9   15.0 /  8.2   46.0 / 20.2
//     12    1  256   10.5 /  7.7   16.2 /  9.2   71.5 / 12.9
//    128    1  128    9.8 /  9.3   12.5 / 10.9   48.6 / 35.7
// One task per wave (a 32-key block or 8 slots) while the workgroups of the call fit the 256 CUs: a step of up to
// 16 KB per CU is a chain of memory latencies, and past one workgroup per CU the parts of a pair only cost their merge.
// Two workgroups per pair pay from windows of 128 keys on (below: 9.9 against 9.5 us at 128 pairs, W = 64).
// A single workgroup of four waves still beats decode_mfma_kernel's two while its cheaper reductions over the query heads
// count and all pairs run at once: from four heads per kv-head, head sizes up to 128, 512 pairs (18.7 / 12.0 at 256 pairs,
// 27.4 / 22.6 at 512 with eight heads; 14.2 / 11.3 and 22.2 / 22.0 with four; 36.9 / 41.9 at 1024).
int split_of(const NhaDecodeArgs* a) {
  const int64_t pairs = (int64_t)a->B * a->H;
  const int tasks = NST + (a->W + 31) / 32, room = (int)(CUS / pairs);
  int P = (tasks + NW - 1) / NW;
  if (P > room) P = room;
  if (P > 2 || (P == 2 && a->W >= 128)) return P;
  return a->K <= 128 && (a->HQ / a->H > 2 || P == 2) && pairs <= 512 ? 1 : 0;
}

template <int D, int G, bool ROT>
int launch(const NhaDecodeArgs* a, int P) {
  constexpr size_t lds = Lds<D, G>::BYTES;
  static std::atomic<bool> configured{false};   // the attribute call is idempotent: a second thread may repeat it
  if (!configured && lds > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)decode_split_kernel<D, G, ROT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      set_error("decode: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
      return NHA_ERR_LAUNCH;
    }
    configured = true;
  }
  SplitArgs sa;
  sa.a = *a;
  sa.P = P;
  const size_t pairs = (size_t)a->B * a->H;
  sa.counter = (int*)a->scratch;
  sa.po = (float*)a->scratch + MAX_SPLIT;
  sa.pml = sa.po + pairs * P * G * D;
  hipLaunchKernelGGL((decode_split_kernel<D, G, ROT>), dim3(a->B * a->H * P), dim3(64 * NW), lds, (hipStream_t)a->stream, sa);
  NHA_CHECK_LAUNCH("nha_decode_step");
  return NHA_OK;
}

template <int D, bool ROT>
int dispatch(const NhaDecodeArgs* a, int G, int P) {
  switch (G) {
    case 1: return launch<D, 1, ROT>(a, P);
    case 2: return launch<D, 2, ROT>(a, P);
    case 4: return launch<D, 4, ROT>(a, P);
    default: return launch<D, 8, ROT>(a, P);
  }
}

}  // namespace

// What any call needs: split_of keeps pairs x workgroups within CUS, and a partial is largest at head size 256 with eight
// heads per kv-head.
size_t decode_scratch_bytes() { return MAX_SPLIT * 4 + (size_t)CUS * (8 * 256 + 2 * 8) * 4; }

// Workgroups per pair at these addresses too; 0 as in split_of.
static int split_at(const NhaDecodeArgs* a) {
  // decode_mfma_kernel reads these (and writes o) element by element, so they may start anywhere; here they move in pieces of
  // up to 16 bytes
  uintptr_t at = reinterpret_cast<uintptr_t>(a->o);
  for (const void* x : {a->q, a->k_pop, a->v_pop, a->g_pop, a->s_pop}) at |= reinterpret_cast<uintptr_t>(x);
  return (at & 15) ? 0 : split_of(a);
}

bool decode_split_uses_scratch(const NhaDecodeArgs* a) { return split_at(a) > 1; }

bool decode_split_wanted(const NhaDecodeArgs* a) {
  const int P = split_at(a);
  return P == 1 || (P > 1 && a->scratch && a->scratch_bytes >= decode_scratch_bytes());
}

int decode_split_impl(const NhaDecodeArgs* a) {
  const int P = split_of(a), G = group_of(a);
  if (a->cos) return a->K == 64 ? dispatch<64, true>(a, G, P) : dispatch<128, true>(a, G, P);
  if (a->K == 256) return dispatch<256, false>(a, G, P);
  return a->K == 64 ? dispatch<64, false>(a, G, P) : dispatch<128, false>(a, G, P);
}

}  // namespace nha
