// Weight gradients of projections that share their input, bf16 in and out, fp32 sums (gfx950): dW_p = dy_p^T x for up to
// four p in one launch, x [T, I], dy_p [T, O_p], dW_p [O_p, I].
//
// The contraction runs over the tokens, the outer axis of both operands, and the outputs are small: 1024 x 1024 from 16384
// tokens is 16 tiles of 256 x 256, so the tokens are split over workgroups (wgrad_split), each leaves its tile's sum in
// fp32 and a second launch adds the splits in a fixed order.  Both operands go to LDS as they lie ([token][column]) and
// are read by the transposing LDS read, which hands a lane the tokens of one column.
//
// Bound: LDS.  A workgroup of eight waves (128 x 64 of the tile each, two per SIMD) reads 197 KB and writes 64 KB of LDS
// per 64 tokens, as many clocks as its matrix products take.  16384 tokens, 1024 columns, outputs of 3 x 1024 + 256: 138 us
// with the sum (0.81 PFLOP/s) against 415 us for four library products, which run 64 x 64 tiles without a split; one output
// of 1024: 54 against 104 us; 2048 columns, 2048 + 2 x 512 + 256: 250 against 468 us.
#include "mfma_common.h"

#include <atomic>

namespace nha {
namespace {
using namespace mf;

constexpr int TW = 256;        // tile: columns of x and of dy
constexpr int TK = 64;         // tokens per step
constexpr int LDW = TW + 16;   // a row is 8 banks past the one before it: the 16 rows of a transposing read meet no conflict
constexpr int NTHR = 512;
constexpr size_t LDS_BYTES = (size_t)4 * TK * LDW * 2;

struct WG {
  const bf16_t* x;
  const bf16_t* dy[4];
  bf16_t* dw[4];
  int O[4], row0[4], tile0[4];   // first row of each output among all of them, first of its column tiles
  int ldy[4];
  int n, T, I, otiles, itiles, split, tsplit, rows;
  float* part;                   // [split][rows][I]
};

__global__ __launch_bounds__(NTHR, 2) void wgrad_kernel(const WG p) {
  extern __shared__ __align__(16) unsigned char smem[];
  lbf16* const tiles = (lbf16*)smem;   // x 0, x 1, dy 0, dy 1
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, kb = lane >> 4;
  // tiles dealt so that an XCD (workgroup id % 8) works on neighbouring tiles of one token range and their rows meet in its L2
  const int total = gridDim.x, per = total >> 3, L = blockIdx.x;
  const int v = L < 8 * per ? (L & 7) * per + (L >> 3) : L;
  const int it = v % p.itiles, ot = (v / p.itiles) % p.otiles, sp = v / (p.itiles * p.otiles);
  int q = 0;
  while (q + 1 < p.n && ot >= p.tile0[q + 1]) ++q;
  const int O = p.O[q], ldy = p.ldy[q], o0 = (ot - p.tile0[q]) * TW, i0 = it * TW;
  const int t0 = sp * p.tsplit, t1 = t0 + p.tsplit < p.T ? t0 + p.tsplit : p.T;
  const int steps = (t1 - t0 + TK - 1) / TK;   // every split holds tokens
  const bf16_t* const xs = p.x + i0;
  const bf16_t* const ys = p.dy[q] + o0;
  const bool whole = i0 + TW <= p.I && o0 + TW <= O;
  const int row = tid >> 5, col = (tid & 31) * 8;   // 16 rows per pass, four passes

  uint4 rx[4], ry[4];
  auto load = [&](int s) {
    const int ts = t0 + s * TK;
    if (whole && ts + TK <= t1) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        rx[u] = *reinterpret_cast<const uint4*>(xs + (int64_t)(ts + 16 * u + row) * p.I + col);
        ry[u] = *reinterpret_cast<const uint4*>(ys + (int64_t)(ts + 16 * u + row) * ldy + col);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = ts + 16 * u + row;
        rx[u] = ry[u] = make_uint4(0, 0, 0, 0);
        if (t < t1 && i0 + col < p.I) rx[u] = *reinterpret_cast<const uint4*>(xs + (int64_t)t * p.I + col);
        if (t < t1 && o0 + col < O) ry[u] = *reinterpret_cast<const uint4*>(ys + (int64_t)t * ldy + col);
      }
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      lds_st16(tiles + buf * TK * LDW + (16 * u + row) * LDW + col, rx[u]);
      lds_st16(tiles + (2 + buf) * TK * LDW + (16 * u + row) * LDW + col, ry[u]);
    }
  };
  const int wi = (wave & 1) * 128, wo = (wave >> 1) * 64;
  f32x4 acc[8][4];
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  load(0);
  store(0);
  if (steps > 1) load(1);
  lds_barrier();
  for (int s = 0; s < steps; ++s) {
    // the other buffer was read in step s - 1, which every wave has left
    if (s + 1 < steps) store((s + 1) & 1);
    if (s + 2 < steps) load(s + 2);
    const lbf16* const X = tiles + (s & 1) * TK * LDW;
    const lbf16* const Y = tiles + (2 + (s & 1)) * TK * LDW;
#pragma unroll
    for (int k = 0; k < TK; k += 32) {
      bf16x8 fy[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) fy[b] = lds_frag_tr(Y, LDW, k, k + 16, wo + 16 * b, lane);
#pragma unroll
      for (int a = 0; a < 8; ++a) {
        const bf16x8 fx = lds_frag_tr(X, LDW, k, k + 16, wi + 16 * a, lane);
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = mfma16(fx, fy[b], acc[a][b]);
      }
    }
    lds_barrier();
  }
  // acc[a][b]: columns i0 + wi + 16 a + 4 kb .. + 4 of row o0 + wo + 16 b + l16
  float* const out = p.part + ((int64_t)sp * p.rows + p.row0[q]) * p.I;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int o = o0 + wo + 16 * b + l16;
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      const int i = i0 + wi + 16 * a + 4 * kb;
      if (o < O && i < p.I) *reinterpret_cast<float4*>(out + (int64_t)o * p.I + i) = make_float4(acc[a][b][0], acc[a][b][1], acc[a][b][2], acc[a][b][3]);
    }
  }
}

// the splits of eight neighbouring elements per thread, added in their order
__global__ __launch_bounds__(256) void wgrad_sum_kernel(const WG p) {
  const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8, plane = (int64_t)p.rows * p.I;
  if (at >= plane) return;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < p.split; ++k) {
    float x[8];
    Elem<float>::ld8(p.part + k * plane + at, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] += x[e];
  }
  const int r = (int)(at / p.I), c = (int)(at % p.I);
  int q = 0;
  while (q + 1 < p.n && r >= p.row0[q + 1]) ++q;
  Elem<bf16_t>::st8(p.dw[q] + (int64_t)(r - p.row0[q]) * p.I + c, s);
}

// Token splits: a round of the chip is 256 workgroups; a step of 64 tokens costs 1.4 us and a workgroup's start and end 6,
// a split's round trip in fp32 its bytes (4 written and 4 read per element) at 4.5 TB/s.
int wgrad_split(int tiles, int T, int64_t elements) {
  const int steps = (T + TK - 1) / TK;
  int best = 1;
  double cost = 1e30;
  for (int s = 1; s <= 32 && s <= steps; ++s) {
    const double rounds = (double)(((int64_t)tiles * s + 255) / 256);
    const double us = rounds * (((steps + s - 1) / s) * 1.4 + 6.0) + s * (double)elements * 8.0 / 4.5e6;
    if (us < cost) {
      cost = us;
      best = s;
    }
  }
  return best;
}

int plan(const NhaWgradArgs* a, WG& p) {
  p.n = a->n; p.T = a->T; p.I = a->I;
  p.otiles = p.rows = 0;
  for (int q = 0; q < a->n; ++q) {
    p.O[q] = a->O[q];
    p.ldy[q] = a->ldy ? a->ldy : a->O[q];
    p.row0[q] = p.rows;
    p.tile0[q] = p.otiles;
    p.rows += a->O[q];
    p.otiles += (a->O[q] + TW - 1) / TW;
  }
  p.itiles = (a->I + TW - 1) / TW;
  const int s = wgrad_split(p.otiles * p.itiles, p.T, (int64_t)p.rows * p.I);
  const int steps = (p.T + TK - 1) / TK;
  p.tsplit = (steps + s - 1) / s * TK;
  p.split = (p.T + p.tsplit - 1) / p.tsplit;   // none of them empty
  return 0;
}

}  // namespace

size_t wgrad_scratch_bytes(const NhaWgradArgs* a) {
  WG p;
  plan(a, p);
  return (size_t)p.split * p.rows * p.I * sizeof(float);
}

int wgrad_impl(const NhaWgradArgs* a) {
  WG p;
  plan(a, p);
  p.x = (const bf16_t*)a->x;
  for (int q = 0; q < a->n; ++q) {
    p.dy[q] = (const bf16_t*)a->dy[q];
    p.dw[q] = (bf16_t*)a->dw[q];
  }
  p.part = (float*)a->scratch;
  static std::atomic<bool> configured{false};   // the attribute call is idempotent: a second thread may repeat it
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute((const void*)wgrad_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES);
    if (e != hipSuccess) {
      set_error("nha_wgrad: cannot reserve %zu bytes of LDS: %s", LDS_BYTES, hipGetErrorString(e));
      return NHA_ERR_LAUNCH;
    }
    configured = true;
  }
  hipStream_t st = (hipStream_t)a->stream;
  hipLaunchKernelGGL(wgrad_kernel, dim3(p.otiles * p.itiles * p.split), dim3(NTHR), LDS_BYTES, st, p);
  const int64_t groups = ((int64_t)p.rows * p.I / 8 + 255) / 256;
  hipLaunchKernelGGL(wgrad_sum_kernel, dim3((unsigned)groups), dim3(256), 0, st, p);
  NHA_CHECK_LAUNCH("nha_wgrad");
  return NHA_OK;
}

}  // namespace nha
