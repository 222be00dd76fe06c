// Shared by the matrix-core decode kernels (decode_mfma.hip, decode_split.hip): vector types, lane helpers, the
// transposing LDS read, streaming loads and the rotate-half of a register pair.
#pragma once
#include "common.h"

namespace nha {
namespace dec {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
#define NHA_LDS __attribute__((address_space(3)))
typedef NHA_LDS bf16_t lbf16;
typedef NHA_LDS float lfloat;

constexpr float LOG2E = 1.4426950408889634f;

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 as_bf16x8(uint4 u) { return __builtin_bit_cast(bf16x8, u); }
__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
// workgroup barrier that orders LDS traffic only; global loads stay in flight across it
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// max over the four 16-lane rows of a wave (lanes l, l^16, l^32, l^48)
__device__ __forceinline__ float max_over_rows(float x) {
  const unsigned u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned v = __float_as_uint(x);
  const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_over_rows(float x) {
  const unsigned u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const unsigned v = __float_as_uint(x);
  const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// the lane (c = l%16, kb = l/16) receives X[4*kb + e][col0 + c] for e = 0..3 and
// X[16 + 4*kb + e][col0 + c] for e = 4..7 of a row-major [32][ld] bf16 LDS tile
__device__ __forceinline__ bf16x8 lds_frag_tr(const lbf16* tile, int ld, int col0, int lane) {
  const int l16 = lane & 15, kb = lane >> 4;
  const lbf16* pa = tile + (4 * kb + (l16 >> 2)) * ld + col0 + 4 * (l16 & 3);
  const lbf16* pb = pa + 16 * ld;
  struct { s16x4 a, b; } t;
  t.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pa);
  t.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pb);
  return __builtin_bit_cast(bf16x8, t);
}

// 16 bytes of a window row: read once per step and never again, so the load is marked
// non-temporal (it does not displace the state lines in L2; measured 145 -> 134 us per step)
__device__ __forceinline__ uint4 ld16_stream(const bf16_t* p) {
  const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  return make_uint4(x[0], x[1], x[2], x[3]);
}

constexpr int MS = 64;   // slots

// rotate-half of the column pair (c, c + D/2), 8 columns at a time: xa holds columns c.., xb columns
// c + D/2..; out_a = xa cos_a - xb sin_a, out_b = xb cos_b + xa sin_b (fp32, rounded to bf16 once)
__device__ __forceinline__ void rope8(uint4& xa, uint4& xb, uint4 ca, uint4 sa, uint4 cb, uint4 sb) {
  const uint32_t a[4] = {xa.x, xa.y, xa.z, xa.w}, b[4] = {xb.x, xb.y, xb.z, xb.w};
  const uint32_t c0[4] = {ca.x, ca.y, ca.z, ca.w}, s0[4] = {sa.x, sa.y, sa.z, sa.w};
  const uint32_t c1[4] = {cb.x, cb.y, cb.z, cb.w}, s1[4] = {sb.x, sb.y, sb.z, sb.w};
  uint32_t oa[4], ob[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float ra[2], rb[2];
#pragma unroll
    for (int hlf = 0; hlf < 2; ++hlf) {
      auto f = [&](uint32_t w) { return __uint_as_float(hlf ? (w & 0xffff0000u) : (w << 16)); };
      ra[hlf] = f(a[i]) * f(c0[i]) - f(b[i]) * f(s0[i]);
      rb[hlf] = f(b[i]) * f(c1[i]) + f(a[i]) * f(s1[i]);
    }
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    bf16x2 pa, pb;
    pa[0] = (__bf16)ra[0]; pa[1] = (__bf16)ra[1];
    pb[0] = (__bf16)rb[0]; pb[1] = (__bf16)rb[1];
    oa[i] = __builtin_bit_cast(uint32_t, pa);
    ob[i] = __builtin_bit_cast(uint32_t, pb);
  }
  xa = make_uint4(oa[0], oa[1], oa[2], oa[3]);
  xb = make_uint4(ob[0], ob[1], ob[2], ob[3]);
}

}  // namespace dec
}  // namespace nha
