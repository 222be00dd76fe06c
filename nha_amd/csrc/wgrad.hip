// Weight gradients of projections that share their input, bf16 in and out, fp32 sums (gfx950): dW_p = dy_p^T x for up to
// four p in one launch, x [T, I], dy_p [T, O_p], dW_p [O_p, I].
//
// The contraction runs over the tokens, the outer axis of both operands, and the outputs are small: 1024 x 1024 from 16384
// tokens is 16 tiles of 256 x 256, so the tokens are split over workgroups (wgrad_split), each leaves its tile's sum in
// fp32 and a second launch adds the splits in a fixed order.  Both operands go straight into LDS as they lie ([token][column],
// LineTile), a ring of four units of 32 tokens, and are read by the transposing LDS read, which hands a lane the tokens of one column.
//
// Bound: the matrix rate that this chip sustains (1.2 PFLOP/s, as a large library product) where the tiles
// fill it, and the fp32 sums' way through memory where few outputs make many splits.  Eight waves hold 128 x 64 of a tile
// each; a unit's fragments are in registers when its products begin and are replaced as they are done with.  Through registers and
// padded rows, two buffers of 64 tokens, no read ahead / now, in turn on one card, with the sum: 16384 tokens, 1024 columns, outputs of
// 3 x 1024 + 256 118 / 112 us (1.0 PFLOP/s; four library products, which run 64 x 64 tiles without a split, 415), one output of 1024 57 / 55
// (library 104); 2048 columns, 2048 + 2 x 512 + 256 221 / 208 (468); 3072 columns, 3072 + 2 x 768 + 512 462 / 429; 4096 tokens, 1024
// columns, 1024 + 2 x 256 + 128 44 / 35.5.  Inside a training step of the layer (8 x 2048 tokens), where the operands come from HBM, both
// launches of each 192 / 182.  A fifth unit in LDS is no faster.
#include "mfma_common.h"

#include <atomic>

namespace nha {
namespace {
using namespace mf;

constexpr int TW = 256;        // tile: columns of x and of dy
constexpr int TK = 32;         // tokens per unit
constexpr int NTHR = 512;
constexpr int NRING = 4;       // units in LDS
typedef LineTile<TW> Tile;     // 32 tokens x 256 columns, 16 KB
constexpr int TBYTES = 2 * Tile::HALF, UNIT = 2 * TBYTES;   // x, then dy
constexpr size_t LDS_BYTES = (size_t)NRING * UNIT;
#define FENCE __builtin_amdgcn_sched_barrier(0)

struct WG {
  const bf16_t* x;
  const bf16_t* dy[4];
  bf16_t* dw[4];
  int O[4], row0[4], tile0[4];   // first row of each output among all of them, first of its column tiles
  int ldy[4];
  int n, T, I, otiles, itiles, split, tsplit, rows;
  float* part;                   // [split][rows][I]
};

__global__ __launch_bounds__(NTHR, 1) void wgrad_kernel(const WG p) {
  extern __shared__ __align__(1024) unsigned char smem[];
  const lbyte* const lds = (const lbyte*)smem;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kb = lane >> 4;
  // tiles dealt so that an XCD (workgroup id % 8) works on neighbouring tiles of one token range and their rows meet in its L2
  const int total = gridDim.x, per = total >> 3, L = blockIdx.x;
  const int v = L < 8 * per ? (L & 7) * per + (L >> 3) : L;
  const int it = v % p.itiles, ot = (v / p.itiles) % p.otiles, sp = v / (p.itiles * p.otiles);
  int q = 0;
  while (q + 1 < p.n && ot >= p.tile0[q + 1]) ++q;
  const int O = p.O[q], ldy = p.ldy[q], o0 = (ot - p.tile0[q]) * TW, i0 = it * TW;
  const int t0 = sp * p.tsplit, t1 = t0 + p.tsplit < p.T ? t0 + p.tsplit : p.T;
  const int units = (t1 - t0 + TK - 1) / TK;   // every split holds tokens
  const bf16_t* const xs = p.x + (int64_t)t0 * p.I + i0;
  const bf16_t* const ys = p.dy[q] + (int64_t)t0 * ldy + o0;

  // LDS-direct loads: block wave + 8 i of a tile's 16, a row and eight columns of it per lane.  Columns past the matrix are read from
  // its last ones (their sums are not stored), tokens past the range from its last one (zeroed in the registers).
  uint32_t xoff[2], yoff[2];   // bytes from the unit's first row
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 16 * i + Tile::load_row(lane), c = (int)Tile::load_col(wave, lane);
    xoff[i] = (uint32_t)(r * p.I + (i0 + c < p.I ? c : p.I - 8 - i0)) * 2;
    yoff[i] = (uint32_t)(r * ldy + (o0 + c < O ? c : O - 8 - o0)) * 2;
  }
  auto issue = [&](int u) {
    const bf16_t* const xb = xs + (int64_t)u * TK * p.I;
    const bf16_t* const yb = ys + (int64_t)u * TK * ldy;
    const uint32_t to = lds0 + (u & (NRING - 1)) * UNIT + Tile::block(0, wave);
    if (t0 + (u + 1) * TK <= t1) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        g2l16(xb, xoff[i], to + Tile::block(i, 0));
        g2l16(yb, yoff[i], to + TBYTES + Tile::block(i, 0));
      }
    } else {
      const int last = t1 - 1 - t0 - u * TK;   // < 31
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 16 * i + Tile::load_row(lane), back = r > last ? r - last : 0;
        g2l16(xb, xoff[i] - (uint32_t)(back * p.I) * 2, to + Tile::block(i, 0));
        g2l16(yb, yoff[i] - (uint32_t)(back * ldy) * 2, to + TBYTES + Tile::block(i, 0));
      }
    }
  };
  // column fragments of the wave's 128 x 64 of the tile: x columns 16 a .., dy columns 16 b ..
  const int wi = (wave & 1) * 128, wo = (wave >> 1) * 64;
  const Tile tile(lds, lane);
  auto xfrag = [&](int u, int a) { return tile.col((uint32_t)((u & (NRING - 1)) * UNIT + wi * 32), a); };
  auto yfrag = [&](int u, int b) { return tile.col((uint32_t)((u & (NRING - 1)) * UNIT + TBYTES + wo * 32), b); };
  f32x4 acc[8][4];
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};

  issue(0);
  if (units > 1) issue(1);
  if (units > 2) issue(2);
  if (units > 2) wait_vm<8>();
  else if (units > 1) wait_vm<4>();
  else wait_vm<0>();
  lds_barrier();
  bf16x8 fx[8], fy[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) fy[b] = yfrag(0, b);
#pragma unroll
  for (int a = 0; a < 8; ++a) fx[a] = xfrag(0, a);
  // A unit's fragments are in registers when its products begin; those of the next one replace them as they are done with, a
  // column block of x (four products) at a time.  One barrier per unit: behind it unit u + 1 has landed for everybody, and
  // everybody has read unit u, so the slot of unit u - 1 takes unit u + 3.
#pragma unroll 1
  for (int u = 0; u + 1 < units; ++u) {
    if (u + 2 < units) wait_vm<4>();
    else wait_vm<0>();
    lds_barrier();
    if (u + 3 < units) issue(u + 3);
    FENCE;
    bf16x8 ny[4];
#pragma unroll
    for (int a = 0; a < 8; ++a) {
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = mfma16(fx[a], fy[b], acc[a][b]);
      FENCE;
      fx[a] = xfrag(u + 1, a);
      if (a % 2 == 0) ny[a / 2] = yfrag(u + 1, a / 2);
      FENCE;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) fy[b] = ny[b];
  }
  const int rem = (t1 - t0) - (units - 1) * TK;   // tokens of the last unit: 4 kb + e and 16 + 4 kb + e in a lane
  if (rem < TK) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bool on = (e < 4 ? 4 * kb + e : 12 + 4 * kb + e) < rem;
#pragma unroll
      for (int a = 0; a < 8; ++a) fx[a][e] = on ? fx[a][e] : (__bf16)0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b) fy[b][e] = on ? fy[b][e] : (__bf16)0.f;
    }
  }
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = mfma16(fx[a], fy[b], acc[a][b]);
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

// Token splits: a round of the chip is 256 workgroups; a unit of 32 tokens costs 0.5 us and a workgroup's start and end 4, a split's round
// trip in fp32 (which mostly stays in the caches) its bytes, 4 written and 4 read per element, at 10 TB/s.  Fitted to the calls' times with 1
// to 32 splits.  With 0.6, 6 and 4.5 TB/s, us before / now: 16384 tokens, 1024 columns, one output of 1024 58.0 (12 splits) / 55.1 (16),
// 12000 47.3 (10) / 43.4 (15), 8192 43.8 (8) / 39.8 (13); 4096, outputs of 1024 + 2 x 256 + 128 38.9 (5) / 35.5 (8).
int wgrad_split(int tiles, int T, int64_t elements) {
  const int steps = (T + TK - 1) / TK;
  int best = 1;
  double cost = 1e30;
  for (int s = 1; s <= 32 && s <= steps; ++s) {
    const double rounds = (double)(((int64_t)tiles * s + 255) / 256);
    const double us = rounds * (((steps + s - 1) / s) * 0.5 + 4.0) + s * (double)elements * 8.0 / 1e7;
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
