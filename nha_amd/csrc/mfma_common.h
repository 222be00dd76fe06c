// Shared by the matrix-core prefill kernels (prefill_mfma.hip, prefill_ring.hip): vector types,
// LDS helpers, the kernel parameter block and the constants of the chunk algebra.
#pragma once
#include "common.h"

namespace nha {
namespace mf {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// explicit LDS address space: keeps every tile access a ds_* instruction (never a flat access)
#define NHA_LDS __attribute__((address_space(3)))
typedef NHA_LDS bf16_t lbf16;
typedef NHA_LDS float lfloat;
typedef NHA_LDS unsigned char lbyte;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void lds_st16(lbf16* p, uint4 v) { *reinterpret_cast<NHA_LDS u32x4*>(p) = (u32x4){v.x, v.y, v.z, v.w}; }
__device__ __forceinline__ float4 lds_ld_f4(const lfloat* p) {
  const f32x4 v = *reinterpret_cast<const NHA_LDS f32x4*>(p);
  return make_float4(v[0], v[1], v[2], v[3]);
}

constexpr int BT = 64;        // chunk rows == window tile keys
constexpr int MS = 64;        // slots
constexpr int GLD = 68;       // LDS row stride (floats) of the gate-cumsum tables
constexpr int SLD = 72;       // LDS row stride (bf16) of the s tables
constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;
// Largest positive decay exponent formed on the MFMA path.  A factor s exp(60) = 1.1e26 still multiplies
// unscaled intra-chunk scores (the layer's default scale is 1) summed over 16 rows with e^28 of fp32
// range to spare; sub-blocks that decay faster are flagged and recomputed exactly.
constexpr float DECAY_CLAMP = 60.f;
// The backward's factored products use one reference per 32-row half of a chunk; the large factor
// s exp(ref - gc_j) <= e^70 = 2.5e30 meets gradient-sized weights there (p (dp - delta), not raw scores), so
// e^18 of fp32 range is enough, and gates drawn as logsigmoid(N(-1, 1)) (32 rows decay by e^-42 +- e^-4.5)
// stay on the matrix-core path; chunks beyond it take the fp32 kernels.
constexpr float BWD_DECAY_CLAMP = 70.f;

struct MP {
  const bf16_t *q_swa, *k_swa, *q_gsa, *k_gsa, *v, *s, *g;
  bf16_t* o;
  float *lse_swa, *lse_gsa;
  const float *h0k, *h0v;
  float *hkt, *hvt;
  const int32_t *cu, *cidx, *coff;
  bf16_t* hkT;   // [NT][H][MS][D]   segment-local chunk-start k-state, transposed ([m][d])
  bf16_t* hvc;   // [NT][H][MS][D]   segment-local chunk-start v-state ([m][d])
  float* gc;     // [NT][H][BT][MS]  chunk-local inclusive gate cumsum
  float* dcum;   // [NT][H][MS]      decay from the segment start to the chunk start
  float *hend_k, *hend_v;   // [NSLOT][H][MS][D]  segment-local end states
  float *hseg_k, *hseg_v;   // [NSLOT][H][MS][D]  true segment-start states
  float* dtot;   // [NSLOT][H][MS]   total decay of a segment
  int* flags;    // [NT][H][4]       per 16-slot block: bit q = sub-block q decays past DECAY_CLAMP
  int T_tot, N, NT, HQ, H, NG, wl, shift;
  int seg_sh;    // a segment is 1 << seg_sh chunks
  int sinks;     // window-only launches (prefill_ring.hip, SINK): zero-logit keys in front of every sequence
  float scale;
};

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 as_bf16x8(uint4 u) { return __builtin_bit_cast(bf16x8, u); }
__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fexp(float x) { return __builtin_amdgcn_exp2f(x * LOG2E); }

__device__ __forceinline__ bf16x8 pack8(f32x4 a, f32x4 b) {
  bf16x8 r;
  r[0] = (__bf16)a[0]; r[1] = (__bf16)a[1]; r[2] = (__bf16)a[2]; r[3] = (__bf16)a[3];
  r[4] = (__bf16)b[0]; r[5] = (__bf16)b[1]; r[6] = (__bf16)b[2]; r[7] = (__bf16)b[3];
  return r;
}

// Tile of a workgroup in a launch of (kv-heads x groups-per-kv-head, chunks) tiles.  Workgroups are dispatched
// in the order L = y * gridDim.x + x and workgroup L runs on XCD L % 8, each XCD with its own L2: XCD k takes
// the k-th eighth of the tile sequence (kv-head, chunk, group of the kv-head), fastest last, so that what an
// XCD works on at one time is a run of neighbouring chunks of one kv-head, whose windows overlap.  Returns the
// tile's x (kv-head * ngrp + group) and y (chunk slot).
__device__ __forceinline__ void xcd_tile(int ngrp, int nchunks, int& vx, int& vy) {
  const int total = gridDim.x * gridDim.y, per = total >> 3;
  const int L = blockIdx.y * gridDim.x + blockIdx.x;
  // the up to seven workgroups beyond a multiple of 8 take the last tiles of the sequence
  const int v = L < 8 * per ? (L & 7) * per + (L >> 3) : L;
  const int g = v % ngrp, rest = v / ngrp;
  vy = rest % nchunks;
  vx = (rest / nchunks) * ngrp + g;
}

// Two chunks of a sequence per workgroup: launch index -> (head x, sequence n, first chunk it of the pair); false for the
// workgroups without one.  The launch (pair_grid) has room for the most pairs that NT chunks in N sequences can make.
// As in xcd_tile XCD k takes the k-th eighth of the sequence (kv-head, pair, head of the kv-head's ngrp), the pairs from the last
// to the first.
// Up to 64 sequences the pairs are counted without gaps, so that the working workgroups come first: left strewn over the launch
// order, those that leave at once give the shader engines unequal shares of the others (2 x 4000 tokens, 4 heads: 256 pairs on 256
// CUs took two rounds).  Each wave counts for itself, a sequence per lane.
// More sequences are not counted, which takes longer the more there are (chunk_nha without / with gradients, 4 heads, W = 512,
// counted / searched: 1000 sequences of 130 tokens 1803 / 1605 and 9435 / 8785 us, 3000 of them 6452 / 5055 and 32437 / 27475):
// sequence n has the places (coff[n] + n) / 2 to (coff[n + 1] + n + 1) / 2, its pairs and where it has an even number of chunks now
// and then one more (every third place of two-chunk sequences, so no engine's in particular), and is found by a search in steps of
// 64.
__device__ __forceinline__ bool pair_tile(const int32_t* coff, int N, int heads, int ngrp, int& x, int& n, int& it) {
  const int lane = threadIdx.x & 63, L = blockIdx.x;
  auto prefix = [&](int c) {   // over the wave, inclusive (DPP: rows of 16 lanes, then across the rows)
    c += __builtin_amdgcn_update_dpp(0, c, 0x111, 0xf, 0xf, false);
    c += __builtin_amdgcn_update_dpp(0, c, 0x112, 0xf, 0xf, false);
    c += __builtin_amdgcn_update_dpp(0, c, 0x114, 0xf, 0xf, false);
    c += __builtin_amdgcn_update_dpp(0, c, 0x118, 0xf, 0xf, false);
    c += __builtin_amdgcn_update_dpp(0, c, 0x142, 0xa, 0xf, false);
    c += __builtin_amdgcn_update_dpp(0, c, 0x143, 0xc, 0xf, false);
    return c;
  };
  int c = 0, incl = 0, total;
  if (N <= 64) {
    c = lane < N ? (coff[lane + 1] - coff[lane] + 1) >> 1 : 0;
    incl = prefix(c);
    total = __builtin_amdgcn_readlane(incl, 63);
  } else {
    total = (coff[N] + N) >> 1;
  }
  const int work = heads * total, per = work >> 3;
  if (L >= work) return false;
  const int v = L < 8 * per ? (L & 7) * per + (L >> 3) : L, g = v % ngrp, rest = v / ngrp;
  x = (rest / total) * ngrp + g;
  const int k = total - 1 - rest % total;
  if (N <= 64) {
    n = __builtin_ctzll(__ballot(k >= incl - c && k < incl));
    it = 2 * (k - __builtin_amdgcn_readlane(incl - c, n));
    return true;
  }
  int step = 64;
  while (step * 64 < N) step *= 64;
  n = 0;   // the first place of sequence n is at k or before, and that of n + 64 step is not
  for (; step; step >>= 6) {
    const int i = n + lane * step;
    const uint64_t before = __ballot(i < N && (coff[i < N ? i : 0] + i) >> 1 <= k);
    n += (__popcll(before) - 1) * step;
  }
  it = 2 * (k - ((coff[n] + n) >> 1));
  return it < coff[n + 1] - coff[n];
}
static inline dim3 pair_grid(int heads, int NT, int N) { return dim3((unsigned)heads * ((unsigned)(NT + N) / 2)); }

// 16 bytes per lane from global memory into LDS at lds_base + 16 * lane (lds_base wave-uniform).
// Issued outside the compiler's memory model: every wait on these loads is written by hand.
__device__ __forceinline__ void g2l16(const void* gbase, uint32_t voff_bytes, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff_bytes), "s"(gbase), "s"(lds_base) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void g2l4(const void* gbase, uint32_t voff_bytes, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff_bytes), "s"(gbase), "s"(lds_base) : "memory");
}

// workgroup barrier that orders LDS traffic only: outstanding global loads (tile prefetches) stay
// in flight across it
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// max over the four 16-lane rows of a wave (lanes l, l^16, l^32, l^48), VALU only
__device__ __forceinline__ float max_over_rows(float x) {
  const unsigned u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned v = __float_as_uint(x);
  const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// A/B fragment of a row-major LDS tile: 8 consecutive elements of row `row` starting at `col`.
__device__ __forceinline__ bf16x8 lds_frag(const lbf16* tile, int ld, int row, int col) {
  return *reinterpret_cast<const NHA_LDS bf16x8*>(tile + row * ld + col);
}

// Transposed fragment of a row-major [rows][ld] bf16 LDS tile: the lane (c = l%16, kb = l/16)
// receives X[r0a + 4*kb + e][col0 + c] for e = 0..3 and X[r0b + 4*kb + e][col0 + c] for e = 4..7.
__device__ __forceinline__ bf16x8 lds_frag_tr(const lbf16* tile, int ld, int r0a, int r0b, int col0, int lane) {
  const int l16 = lane & 15, kb = lane >> 4;
  const lbf16* pa = tile + (r0a + 4 * kb + (l16 >> 2)) * ld + col0 + 4 * (l16 & 3);
  const lbf16* pb = tile + (r0b + 4 * kb + (l16 >> 2)) * ld + col0 + 4 * (l16 & 3);
  struct { s16x4 a, b; } t;
  t.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pa);
  t.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pb);
  return __builtin_bit_cast(bf16x8, t);
}

// A 32-row bf16 tile in LDS that LDS-direct loads fill and both row fragments and transposing reads take at the LDS's full rate.
// Blocks of 16 rows x 32 columns (1 KB, one load of a wave, four neighbouring lanes 64 consecutive bytes of a row); the
// 16-byte piece c of row r lies at piece c ^ f(r) of its 64 bytes, f(r) = -(r / 4) mod 4.  Cycles of a wave instruction (eight waves):
// row fragment 4.1, transposing read 3.2; with f(r) = r / 4, 8.1 and 4.5.
// What neighbouring lanes cover decides the rate of the loads: out of L2 a CU pulls 38 GB/s in 16-byte pieces of 16 rows, 74 in 32-byte
// pieces, 135 in 64-byte and 133 in 128-byte rows; all 256 together 9.4, 18.0, 20.5 and 30.1 TB/s.
template <int D>
struct LineTile {
  static constexpr int HALF = D / 32 * 1024;   // bytes of 16 rows
  static __device__ __forceinline__ int f(int r) { return -(r >> 2) & 3; }
  // loads: where the block of rows 16 rh .. and columns 32 cb .. lies; the row of it that a lane takes eight columns of, and the
  // first of them
  static __device__ __forceinline__ uint32_t block(int rh, int cb) { return (uint32_t)(rh * HALF + cb * 1024); }
  static __device__ __forceinline__ int load_row(int lane) { return lane >> 2; }
  static __device__ __forceinline__ uint32_t load_col(int cb, int lane) { return (uint32_t)(32 * cb + 8 * ((lane & 3) ^ f(lane >> 2))); }
  // reads: byte offsets of a lane's part of a row fragment and of a transposing read of even / odd 16-column blocks
  static __device__ __forceinline__ uint32_t row_at(int lane) {
    const int l16 = lane & 15, kb = lane >> 4;
    return (uint32_t)(l16 * 64 + (kb ^ f(l16)) * 16);
  }
  static __device__ __forceinline__ uint32_t col_at(int lane) {
    const int l16 = lane & 15, r = 4 * (lane >> 4) + (l16 >> 2);
    return (uint32_t)(r * 64 + (((l16 >> 1) & 1) ^ f(r)) * 16 + (l16 & 1) * 8);
  }
  const lbyte* lds;
  uint32_t ra, ca;
  __device__ __forceinline__ LineTile(const lbyte* l, int lane) : lds(l), ra(row_at(lane)), ca(col_at(lane)) {}
  // row fragment of the tile at byte address a (a multiple of 64): row 16 rh + l16, columns 32 ks + 8 kb ..
  __device__ __forceinline__ bf16x8 row(uint32_t a, int rh, int ks) const {
    return *reinterpret_cast<const NHA_LDS bf16x8*>(lds + (a + ra) + rh * HALF + ks * 1024);
  }
  // transposed fragment: X[4 kb + e][16 c + l16] (e < 4) and X[16 + 4 kb + e - 4][..]
  __device__ __forceinline__ bf16x8 col(uint32_t a, int c) const {
    const lbyte* pa = lds + ((a + ca) ^ ((c & 1) * 32)) + (c >> 1) * 1024;
    struct { s16x4 a, b; } t;
    t.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pa);
    t.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)(pa + HALF));
    return __builtin_bit_cast(bf16x8, t);
  }
};

// the slot recurrence is cut into segments of 1 << sh <= SEG chunks (two-level state pass; prefill_mfma.hip: plan_scratch)
constexpr int SEG = 8;

__device__ __forceinline__ int seg_slot(const int32_t* coff, int n, int it, int sh) { return (coff[n] >> sh) + (it >> sh) + n; }

// decay-factor fragments of the slot branch, built once per workgroup in MFMA operand order
constexpr int NSEA = 24;   // fragments s*decay with rows = slots  (A operand of the logit update)
constexpr int NSEB = 20;   // fragments s*decay with rows = tokens (A operand of the slot-read weights)
__device__ __forceinline__ int sea_base(int Q) { return Q == 0 ? 0 : Q == 1 ? 4 : Q == 2 ? 8 : 16; }
__device__ __forceinline__ int seb_base(int Q) { return Q == 0 ? 0 : Q == 1 ? 2 : Q == 2 ? 6 : 12; }

}  // namespace mf

// prefill_mfma.hip: the workgroups of level 2 of the forward's state pass in one launch, 0 where it takes two
int64_t state_link_grid(int NT, int N, int H, int D, int seg_sh);
// the state pass in segment form
int prefill_mfma_segment_states(const NhaPrefillArgs* a, mf::MP* out);
// prefill_bwd_slot.hip: the slot branch of the backward but for the carried state gradient, from a state pass in segment form; in
// how many parts the query heads of a kv-head are summed, each part's sums of its own after those of the one before
int bwd_slot_parts(const NhaPrefillBwdArgs* a);
int bwd_slot_branch(const NhaPrefillBwdArgs* a, const mf::MP& m, float* delta, float* xg, float* dsi, float* ek, float* ev, float* dks,
                    float* dvs, int parts);
// output pass with LDS-direct window loads (prefill_ring.hip); false when the shape is not served
bool prefill_ring_supported(const mf::MP& p, int D);
int prefill_ring_launch(const mf::MP& p, int D, hipStream_t st);
bool prefill_ring_raw(int HQ, int NT);   // whether its queries are not scaled before the products

// the same for head size 256, one query head per workgroup (prefill_ring256.hip)
bool prefill_ring256_supported(const mf::MP& p, int D);
int prefill_ring256_launch(const mf::MP& p, hipStream_t st);

}  // namespace nha
