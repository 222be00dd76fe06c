// Output pass of the bf16 matrix-core prefill at head size 256 (K == V == 256, M == 64), one query head
// per workgroup: the data movement and loop of prefill_ring.hip (operands straight from global memory
// into LDS, the window walked first in 32-key units, the slot branch folded into the running softmax
// afterwards; chunk algebra of nha_fla/ops/nha/chunk_fused.py:186-283, one softmax over
// [slots | window] as in nha_fla/ops/nha/chunk.py:459-470) re-proportioned for rows of 512 bytes:
//
//  * One workgroup = NCH consecutive 64-row chunks of a sequence for one query head, 4 NCH waves of 16 query
//    rows: the accumulators of 16 rows x 256 columns are 64 registers, those of 32 rows would not leave room
//    for the fragments.  Launched with NCH = 2: the two chunks walk one window (20 units at a window of 512
//    where two workgroups of one chunk fetch 18 each) with two waves per SIMD.
//  * A unit of 32 keys is 16 KB of K and 16 KB of V.  K and V units live in two rings of three buffers
//    with their own schedules: iteration u forms the scores of unit u + 1 and the products of unit u, so
//    after its barrier the K buffer of unit u + 1 and the V buffer of unit u - 1 are free and take K of
//    unit u + 4 and V of unit u + 2; both have two iterations to land.
//    An iteration that does nothing else has its loads between the products and steps two pointers; with each request's
//    address formed anew it took 2400 cycles, now 2100, 1056 of them matrix instructions (kernel, 32768 tokens packed, 4 heads,
//    W = 512: 205 -> 198 us; 8 x 2048 tokens 89.5 -> 86.6).
//  * Query rows go through LDS in whole lines (a fragment as it lies in memory is 16 bytes of 16 rows: 56 cycles a load, a line
//    load 16), unscaled, the scores taking the scale as they take the reference (198 -> 193 us; 86.6 -> 85.0).
//  * Fragments are read from LDS a few matrix instructions before their use and not earlier: sixteen K
//    and sixteen V fragments held at once (128 registers) would push the accumulators out of the
//    register file.
//  * The slot branch passes its tiles (k-state, k_gsa rows, v-state, v rows: 32 KB each a chunk) through four ring buffers, one
//    kind at a time for both chunks together, so that all eight waves work on their own rows; the second chunk's decay tables
//    take the two buffers left.  The k-states are requested into the buffers that the last iterations of the loop retire, every
//    further tile when all waves are done with the one before, and what needs no tile (tables, softmax, weights) is computed
//    while it is on its way.  (Chunk by chunk, with half of the waves idle, the branch took 34 of a workgroup's 100 thousand
//    cycles, now 21: 213 -> 205 us, 93.0 -> 89.5.)
//  * The softmax reference of a row is fixed by the prologue (the chunk's own keys): rescaling 64
//    accumulator registers inside the loop costs the loop its registers whether or not the branch is
//    taken.  A unit whose maximum tops the reference by 2^96 hands the wave's 16 rows to the exact pass
//    (prefill_exact.h) and is clamped.
#include "prefill_exact.h"

#include <mutex>
#include <type_traits>

namespace nha {
namespace {
using namespace mf;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

#define NHA_FENCE() __builtin_amdgcn_sched_barrier(0)
#define NHA_PIN(x) asm volatile("" : "+v"(x))

__device__ __forceinline__ unsigned cvt2(float a, float b) {
  bf16x2 t;
  t[0] = (__bf16)a;
  t[1] = (__bf16)b;
  return __builtin_bit_cast(unsigned, t);
}

template <int NCH>
struct Cfg {
  static constexpr int D = 256;
  static constexpr int KS = D / 32;            // 32-column blocks per row == contraction steps of q.k
  static constexpr int DB = D / 16;            // 16-row blocks of O^T
  static constexpr int UB = 32 * D * 2;        // bytes of a 32-row unit buffer (16 KB)
  static constexpr int HB = UB / 2;            // bytes of its 16-row half
  static constexpr int NR = 3;                 // buffers per ring
  static constexpr int NW = 4 * NCH;           // waves: four 16-row sub-blocks per chunk
  static constexpr int BPU = 2 * KS;           // 1 KB blocks of a unit buffer (16)
  static constexpr int LPB = BPU / NW;         // LDS-direct loads per wave for one buffer (4 or 2)
  static constexpr int RING_K = 0, RING_V = NR * UB;
  static constexpr int GC = 2 * NR * UB;       // gate cumsum fp32 [64][64], pieces XORed with row % 16
  static constexpr int SS = GC + 16384;        // s bf16 [64][64], pieces XORed with row % 8
  static constexpr int ETAB = SS + 8192;       // decay tables, 6 units of 4 KB
  static constexpr int GC2 = ETAB + 6 * 4096;  // gate cumsums of the second chunk (NCH == 2)
  static constexpr int USED = GC2 + (NCH - 1) * 16384, EXACT = ExactSmem<D, NCH, true>::bytes;
  static constexpr int BYTES = USED > EXACT ? USED : EXACT;
};

// LDS layout of a 32-row buffer: LineTile.
template <int NCH>
__global__ __launch_bounds__(256 * NCH, 1) void ring256_out_kernel(const MP p) {
  using C = Cfg<NCH>;
  constexpr int XB0 = 64 * NCH - 32;           // first key of unit 0, relative to the workgroup's first row
  constexpr int D = C::D, KS = C::KS, DB = C::DB, UB = C::UB, HB = C::HB, NR = C::NR, NW = C::NW, LPB = C::LPB;
  extern __shared__ __align__(1024) unsigned char smem_[];
  lbyte* const lds = (lbyte*)smem_;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kb = lane >> 4;
  const int H = p.H, HQ = p.HQ, NG = p.NG;
  // tiles dealt so that an XCD works on neighbouring chunks of one kv-head (xcd_tile, pair_tile); chunks from the last to the first
  int vx, chunk, n, it;
  if constexpr (NCH == 1) {
    int vy;
    xcd_tile(NG, p.NT, vx, vy);
    chunk = p.NT - 1 - vy;
    n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  } else {
    if (!pair_tile(p.coff, p.N, p.HQ, NG, vx, n, it)) return;
    chunk = p.coff[n] + it;
  }
  const int hq = vx, h = hq / NG;
  const int ch = wave >> 2;                    // this wave's chunk of the workgroup's NCH
  const int Q = wave & 3;                      // its 16-row sub-block of that chunk
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int c0 = bos + it * BT;                // first row of the workgroup (its first chunk)
  const int rows_wg = (eos - c0) < NCH * BT ? (eos - c0) : NCH * BT;
  const int rows = rows_wg - BT * ch < 0 ? 0 : (rows_wg - BT * ch < BT ? rows_wg - BT * ch : BT);   // rows of this wave's chunk
  const float cs = p.scale * LOG2E;
  const int64_t cg = (int64_t)chunk * H + h;   // (chunk, kv-head) of the first chunk; the second one is H further
  const int irow = 16 * Q + l16;               // this lane's query row inside its chunk
  const int yrow = BT * ch + irow;             // ... and inside the workgroup's rows
  // per chunk of the workgroup, the 16-row blocks that are formed again at the end: those that decay too fast for the split decay
  // (flags of the state pass), and in the waves' own words those whose scores leave the range of their softmax reference
  int exact[NCH], bad = 0;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    exact[c] = 0;
    if (rows_wg > BT * c) {
      const int* const f = p.flags + (cg + (int64_t)c * H) * 4;
      exact[c] = f[0] | f[1] | f[2] | f[3];
    }
  }
  const int r0w = BT * ch + 16 * Q;            // first row of this wave

  // window units: unit u covers keys [c0 + XB0 - 32 u, c0 + XB0 + 32 - 32 u); c0 - bos is a multiple of 64, so no
  // unit starts before its sequence; units 0 .. 2 NCH - 1 are the workgroup's own rows and may run past eos
  int lowest = bos;
  if (p.wl >= 0 && c0 - p.wl > bos) lowest = c0 - p.wl;
  const int nunits = (c0 + BT * NCH - lowest + 31) / 32;   // >= 2 NCH

  // ---- LDS-direct loads: block b = wave + NW i of a buffer; per lane a row of the block and a 16-byte piece
  const int lrow = LineTile<D>::load_row(lane);
  // one 32-row buffer from rows of `src` (row stride in elements): row r of the buffer is global row rowmap(r)
  auto issue_buffer = [&](uint32_t lds_buf, const bf16_t* src, uint32_t stride, auto rowmap) {
#pragma unroll
    for (int i = 0; i < LPB; ++i) {
      const int b = wave + NW * i;           // < 16
      const int rh = b / KS, cq = b % KS;
      const int r = 16 * rh + lrow;
      const uint32_t off = ((uint32_t)rowmap(r) * stride + LineTile<D>::load_col(cq, lane)) * 2;
      g2l16(src, off, lds0 + lds_buf + rh * HB + cq * 1024);
    }
  };
  const bf16_t* const kbase = p.k_swa + ((int64_t)bos * H + h) * D;
  const bf16_t* const vbase = p.v + ((int64_t)bos * H + h) * D;
  // rows past eos (the workgroup's own units only) are read from row eos - 1: always masked, always finite
  auto unit_row = [&](int u) {
    const int key0 = c0 + XB0 - 32 * u - bos;
    const int last = eos - 1 - bos;
    return [=](int r) { return key0 + r < last ? key0 + r : last; };
  };
  auto issue_k = [&](int u, uint32_t slot_off) { issue_buffer(C::RING_K + slot_off, kbase, (uint32_t)(H * D), unit_row(u)); };
  auto issue_v = [&](int u, uint32_t slot_off) { issue_buffer(C::RING_V + slot_off, vbase, (uint32_t)(H * D), unit_row(u)); };
  // units >= 2 NCH lie wholly before the workgroup's rows (never past eos): fixed per-lane offsets from a wave-uniform row pointer
  uint32_t uoff[LPB], boff[LPB];
#pragma unroll
  for (int i = 0; i < LPB; ++i) {
    const int b = wave + NW * i;
    const int rh = b / KS, cq = b % KS;
    uoff[i] = ((uint32_t)(16 * rh + lrow) * (uint32_t)(H * D) + LineTile<D>::load_col(cq, lane)) * 2;
    boff[i] = lds0 + rh * HB + cq * 1024;
  }

  auto tok_from = [&](int gs, int r) {   // source token of row r of a chunk whose row 0 has source token gs, kept inside the sequence
    int t = gs + r;
    t = t < bos ? bos : t;
    t = t < eos ? t : eos - 1;
    return t - bos;
  };
  // gate cumsums of chunk c of the workgroup (16 blocks of 4 rows; rows past the chunk's last were never written by the
  // state pass and stay unused) and the s rows of its source tokens
  auto issue_gc = [&](int c_, uint32_t dst) {
#pragma unroll
    for (int i = 0; i < 16 / NW; ++i) {
      const int b = wave + NW * i;
      const int r = 4 * b + (lane >> 4);
      const int c = (lane & 15) ^ (r & 15);
      g2l16(p.gc + (cg + (int64_t)c_ * H) * BT * MS, (uint32_t)(r * MS + 4 * c) * 4, lds0 + dst + b * 1024);
    }
  };
  auto issue_s = [&](int gs) {
#pragma unroll
    for (int i = 0; i < 8 / NW; ++i) {
      const int b = wave + NW * i;
      const int r = 8 * b + (lane >> 3);
      const int c = (lane & 7) ^ (r & 7);
      g2l16(p.s + ((int64_t)bos * H + h) * MS, ((uint32_t)tok_from(gs, r) * (uint32_t)(H * MS) + (uint32_t)c * 8) * 2, lds0 + C::SS + b * 1024);
    }
  };

  auto gc_at = [&](uint32_t gco, int j, int m) -> const lfloat* { return (const lfloat*)(lds + gco + j * 256 + (((m >> 2) ^ (j & 15)) * 16) + (m & 3) * 4); };
  auto s_at = [&](int j, int m) -> const lbf16* { return (const lbf16*)(lds + C::SS + j * 128 + (((m >> 3) ^ (j & 7)) * 16) + (m & 7) * 2); };
  // decay tables E_Q[j][m] = s_j[m] exp(min(gr_Q[m] - gc_j[m], DECAY_CLAMP)) for the rows j of the 16-row
  // blocks jb <= Q, zero elsewhere (gr_Q: gate cumsum of the row before sub-block Q, 0 for Q = 0); rows
  // whose source token does not exist carry no weight.  32-row units (64 columns) in blocks of 16 rows x 32
  // columns, two planes of 32-byte rows each, which is what the transposing read takes:
  // E_0 -> unit 0, E_1 -> 1, E_2 -> 2,3, E_3 -> 4,5; a thread makes 8 consecutive slots of a row.
  // (of chunk c_ of the workgroup, from its gate cumsums at gco and the s rows at SS, to two places)
  auto build_decay_tables = [&](int c_, uint32_t gco, uint32_t to03, uint32_t to45) {
    // first row whose source token exists, number of rows; rows outside carry no weight
    const int vlo = (p.shift - (it + c_) * BT) < 0 ? 0 : (p.shift - (it + c_) * BT);
    const int rows_c = rows_wg - c_ * BT < BT ? rows_wg - c_ * BT : BT;
    for (int item = tid; item < 6 * 256; item += 64 * NW) {
      const int U = item >> 8, r32 = (item >> 3) & 31, m = (item & 7) * 8;
      const int Qt = U == 0 ? 0 : U == 1 ? 1 : U < 4 ? 2 : 3;
      const int pr = (U == 3 || U == 5) ? 1 : 0;
      const int j = 32 * pr + r32;
      const bool ok = (j >> 4) <= Qt && j >= vlo && j < rows_c;
      bf16x8 out;
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = (__bf16)0.f;
      if (ok) {
        f32x4 gv[2], gr[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          gv[hh] = *reinterpret_cast<const NHA_LDS f32x4*>(gc_at(gco, j, m + 4 * hh));
          gr[hh] = (f32x4){0.f, 0.f, 0.f, 0.f};
          if (Qt > 0) gr[hh] = *reinterpret_cast<const NHA_LDS f32x4*>(gc_at(gco, 16 * Qt - 1, m + 4 * hh));
        }
        const bf16x8 sv = *reinterpret_cast<const NHA_LDS bf16x8*>(s_at(j, m));
#pragma unroll
        for (int e = 0; e < 8; ++e) out[e] = (__bf16)((float)sv[e] * fexp(fminf(gr[e >> 2][e & 3] - gv[e >> 2][e & 3], DECAY_CLAMP)));
      }
      const uint32_t unit = (U < 4 ? to03 : to45 - 4 * 4096) + U * 4096, block = (r32 >> 4) * 2048 + (m >> 5) * 1024;
      *reinterpret_cast<NHA_LDS bf16x8*>(lds + unit + block + ((m >> 4) & 1) * 512 + (r32 & 15) * 32 + (m & 15) * 2) = out;
    }
  };
  // ---- requests: the gate blocks and the window queries, these through the rings in whole lines (a fragment loaded from global
  //      memory as it is, 16 bytes of 16 rows, takes three times as long); then K and V of the first units, under way while the
  //      decay tables are built, and the second chunk's gate cumsums, which wait in a place of their own ------------------
  const bool second = rows_wg > BT;   // the workgroup has a second chunk
  issue_gc(0, C::GC);
  issue_s(c0 - p.shift);
#pragma unroll
  for (int j = 0; j < NW / 2; ++j)    // rows past the end of the sequence: its last, zeroed once they are in their registers
    issue_buffer(j * UB, p.q_swa + ((int64_t)c0 * HQ + hq) * D, (uint32_t)(HQ * D), [&](int r) { return 32 * j + r < rows_wg ? 32 * j + r : rows_wg - 1; });
  const uint32_t kaddr = LineTile<D>::row_at(lane), vaddr = LineTile<D>::col_at(lane);
  // row fragment (rows 16 kk + l16 of a buffer, columns 32 ks + 8 kb ..) of a buffer at byte address a
  auto kfrag = [&](uint32_t a, int kk, int ks) -> bf16x8 {
    const lbyte* base = lds + (a + kaddr);     // one address per buffer; the fragment is a constant offset from it
    return *reinterpret_cast<const NHA_LDS bf16x8*>(base + (kk * HB + ks * 1024));
  };
  wait_vm<0>();
  lds_barrier();
  bf16x8 qs[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    // rows that do not exist score 0: scores of a copied row could top the reference below and flag rows of another sequence
    const u32x4 x = __builtin_bit_cast(u32x4, kfrag(wave * HB, 0, ks));
    qs[ks] = __builtin_bit_cast(bf16x8, irow < rows ? x : (u32x4){0u, 0u, 0u, 0u});
  }
  lds_barrier();
  issue_k(0, 0);
  issue_v(0, 0);
  issue_k(1, UB);
  issue_v(1, UB);
  if (2 < nunits) issue_k(2, 2 * UB);
  if (NCH == 2 && second) issue_gc(1, C::GC2);
  build_decay_tables(0, C::GC, C::ETAB, C::ETAB + 4 * 4096);
  NHA_FENCE();

  // ---- window loop state ------------------------------------------------------------------------
  f32x4 O[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) O[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
  f32x4 Lw = {0.f, 0.f, 0.f, 0.f};
  float nm = 0.f;                      // minus the running reference maximum, log2 units
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;
  constexpr float THR = 8.f;           // the reference moves (prologue, slot branch) when a score tops it by more than 2^THR
  constexpr float BIG = 96.f;          // scores this far above the reference leave the matrix-core path

  // transposed fragment of a buffer: X[4 kb + e][16 db + l16] (e < 4) and X[16 + 4 kb + e - 4][..]
  auto vfrag = [&](uint32_t a, int db) -> bf16x8 {
    const lbyte* base = lds + ((a + vaddr) ^ ((db & 1) * 32));   // two addresses per buffer
    const lbyte* pa = base + (db >> 1) * 1024;
    struct { s16x4 a, b; } t;
    t.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pa);
    t.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)(pa + HB));
    return __builtin_bit_cast(bf16x8, t);
  };
  auto mask_unit = [&](f32x4 (&S)[2], int u) {
    const int xbase = XB0 - 32 * u;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = xbase + 16 * kk + 4 * kb + r;
        const bool ok = (x <= yrow) && (p.wl < 0 || x >= yrow - p.wl);
        if (!ok) S[kk][r] = -INFINITY;
      }
  };
  // a unit needs the mask when its last key lies after this wave's first row or its first key before the window of
  // this wave's last row
  auto is_edge = [&](int u) -> bool { return (XB0 + 31 - 32 * u > r0w) || (p.wl >= 0 && XB0 - 32 * u < r0w + 15 - p.wl); };

  // the reference moves up by delta: everything accumulated so far shrinks by 2^-delta
  auto rescale_acc = [&](float delta) {
    const float alpha = fexp2(-delta);
    nm -= delta;
#pragma unroll
    for (int r = 0; r < 4; ++r) Lw[r] *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) O[db][r] *= alpha;
  };
  auto rescale = [&](f32x4 (&S)[2], float rmax) {
    const float delta = fmaxf(max_over_rows(rmax), 0.f);
    rescale_acc(delta);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[kk][r] -= delta;
  };
  auto max8 = [&](const f32x4 (&S)[2]) -> float {
    const float a = fmaxf(fmaxf(S[0][0], S[0][1]), fmaxf(S[0][2], S[0][3]));
    return fmaxf(a, fmaxf(fmaxf(S[1][0], S[1][1]), fmaxf(S[1][2], S[1][3])));
  };

  f32x4 Sc[2], Sn[2];
  // fragments requested from LDS ahead of the matrix instruction that takes them: with one wave per SIMD 4 to 14 measure
  // the same; with two (the other wave fills the waits) 2 is best by 1.5 % (1, 3, 4: 0 - 1 %; 8, 10: slower)
  constexpr int PD = NCH == 2 ? 2 : 6;
  // ---- prologue: scores of unit 0, K fragments of unit 1 -----------------------------------------------
  wait_vm<0>();
  lds_barrier();
  {
    Sc[0] = (f32x4){0.f, 0.f, 0.f, 0.f};
    Sc[1] = Sc[0];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      Sc[0] = mfma16(kfrag(C::RING_K, 0, ks), qs[ks], Sc[0]);
      Sc[1] = mfma16(kfrag(C::RING_K, 1, ks), qs[ks], Sc[1]);
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int r = 0; r < 4; ++r) Sc[kk][r] *= cs;
    mask_unit(Sc, 0);   // unit 0 is always an edge unit
    const float x = max8(Sc);
    if (__any(x > THR)) rescale(Sc, x);
  }
  // every wave has read the K buffer of unit 0: unit 3 takes it; every wave has built its part of the first chunk's
  // decay tables, the last readers of its s rows: the second chunk's s rows take their place (one load per wave,
  // older than everything the loop's waits leave in flight)
  lds_barrier();
  if (NCH == 2 && second) issue_s(c0 + BT - p.shift);
  if (3 < nunits) issue_k(3, 0);

  // slot-branch queries, requested while the last unit is worked on: whole lines, as 1 KB blocks of 16 rows x 32 columns, put
  // into fragment order through LDS when they are taken
  uint4 qraw[KS];
  auto load_qg = [&]() {
    const int y = BT * ch + 16 * Q + lrow;
    const bf16_t* qp = p.q_gsa + ((int64_t)(c0 + (y < rows_wg ? y : rows_wg - 1)) * HQ + hq) * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qraw[ks] = *reinterpret_cast<const uint4*>(qp + LineTile<D>::load_col(ks, lane));
  };
  bf16x8 qg[KS];
  auto take_qg = [&](uint32_t buf) {   // (two blocks per wave: what a wave writes there it alone reads)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const uint32_t at = buf + wave * 2048 + (ks & 1) * 1024;
      *reinterpret_cast<NHA_LDS u32x4*>(lds + (at + lane * 16)) = __builtin_bit_cast(u32x4, qraw[ks]);
      qg[ks] = *reinterpret_cast<const NHA_LDS bf16x8*>(lds + (at + kaddr));
    }
  };
  auto pack_p = [&]() -> bf16x8 {
    const u32x4 t = {cvt2(Sc[0][0], Sc[0][1]), cvt2(Sc[0][2], Sc[0][3]), cvt2(Sc[1][0], Sc[1][1]), cvt2(Sc[1][2], Sc[1][3])};
    bf16x8 P = __builtin_bit_cast(bf16x8, t);
    NHA_PIN(P);
    return P;
  };

  // The slot branch takes four tiles of 64 rows per chunk (k-state, k_gsa rows, v-state, v rows), one after the other and those of
  // all NCH chunks together, each as two 32-row halves in ring buffers.  With at least five units the buffers that the window
  // loop retires last take the halves of the k-states while it still runs (a half is as many loads as a unit buffer, so the
  // in-flight counts of the loop stay what they are); shorter windows request them afterwards.
  const bf16_t* const t_kg = p.k_gsa + ((int64_t)bos * H + h) * D;
  auto issue_ta = [&](uint32_t off, int c_, int half) { issue_buffer(off, p.hkT + (cg + (int64_t)c_ * H) * MS * D, (uint32_t)D, [=](int r) { return 32 * half + r; }); };
  auto issue_tb = [&](uint32_t off, int c_, int half, const bf16_t* src) {   // rows of the source tokens of a chunk
    issue_buffer(off, src, (uint32_t)(H * D), [&](int r) { return tok_from(c0 + c_ * BT - p.shift, 32 * half + r); });
  };
  auto issue_tc = [&](uint32_t off, int c_, int half) { issue_buffer(off, p.hvc + (cg + (int64_t)c_ * H) * MS * D, (uint32_t)D, [=](int r) { return 32 * half + r; }); };
  const bool early = nunits >= 5;
  const int last_c = NCH == 2 && second ? 1 : 0;   // (a workgroup of one chunk requests that chunk's twice)
  uint32_t oT[NCH][2];   // where the halves of a chunk's tile lie: the K buffers, and a V buffer
  oT[0][0] = C::RING_K, oT[0][1] = C::RING_K + UB;
  if constexpr (NCH == 2) oT[1][0] = C::RING_K + 2 * UB, oT[1][1] = C::RING_V;
  uint32_t oE2 = C::RING_V + UB, oE2b = C::RING_V + 2 * UB;   // the two buffers left, which take the second chunk's decay tables
  // ring positions as rotating buffer offsets: s0 = buffer of unit u, s1 of unit u+1, s2 of unit u+2
  uint32_t s0 = 0, s1 = UB, s2 = 2 * UB;
  // K of unit u + 4 and V of unit u + 2
  const bf16_t *kp = p.k_swa + (((int64_t)c0 + XB0 - 32 * 4) * H + h) * D, *vp = p.v + (((int64_t)c0 + XB0 - 32 * 2) * H + h) * D;
  const int64_t upr = (int64_t)32 * H * D;
  auto step = [&](int u, auto body_) {
    constexpr bool BODY = decltype(body_)::value;
    const uint32_t k_n = C::RING_K + s1;    // K of unit u+1
    const uint32_t v_c = C::RING_V + s0;    // V of unit u
    // ---- phase A: scores of unit u+1 on the matrix core (two accumulators in turn), exponentials of
    //      unit u on the VALU (one per two products); K fragment i = 2 ks + kk is read PD products ahead ----
    bf16x8 kfr[2 * KS];
    NHA_FENCE();
#pragma unroll
    for (int i = 0; i < PD; ++i) kfr[i] = kfrag(k_n, i & 1, i >> 1);
    NHA_FENCE();
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
      const int ks = i >> 1, kk = i & 1;
      if (i + PD < 2 * KS) kfr[i + PD] = kfrag(k_n, (i + PD) & 1, (i + PD) >> 1);
      Sn[kk] = mfma16(kfr[i], qs[ks], ks == 0 ? (f32x4){0.f, 0.f, 0.f, 0.f} : Sn[kk]);
      if (kk == 1) {
        Sc[ks >> 2][ks & 3] = fexp2(Sc[ks >> 2][ks & 3]);
        NHA_PIN(Sc[ks >> 2][ks & 3]);
      }
      NHA_FENCE();
    }
    const bf16x8 Pq = pack_p();
    NHA_FENCE();
    // K of unit u+2 and V of unit u (requested two iterations ago) have landed for this wave, then for
    // everybody.  What may stay in flight: the requests of the previous iteration.
    if constexpr (BODY) {
      wait_vm<2 * LPB>();
    } else if (u >= 1) {
      if (early) {                    // every iteration requests two buffers' worth, V side first
        if (u + 2 == nunits) wait_vm<LPB>();   // last iteration: also V of the last unit; the tile half behind it may fly
        else wait_vm<2 * LPB>();
      } else {
        wait_vm<0>();
      }
    }
    lds_barrier();
    if constexpr (!BODY) {
      if (u + 2 < nunits) {
        issue_v(u + 2, s2);
      } else if (NCH == 2 && early) {
        oT[NCH - 1][1] = C::RING_V + s2;
        issue_ta(oT[NCH - 1][1], last_c, 1);
      }
      if (u + 4 < nunits) {
        issue_k(u + 4, s1);   // unit u+4 takes the buffer of unit u+1
      } else if (early) {
        const uint32_t off = C::RING_K + s1;
        if (u + 4 == nunits) {
          oT[0][0] = off;
          issue_ta(off, 0, 0);
        } else if (u + 3 == nunits) {
          oT[0][1] = off;
          issue_ta(off, 0, 1);
        } else if (NCH == 2) {
          oT[NCH - 1][0] = off;
          issue_ta(off, last_c, 0);
        }
      }
    }
    auto request = [&](int i) {   // in the common form the loads stand between the products of phase B, V first
      if constexpr (BODY) {
        if (i < LPB) g2l16(vp, uoff[i], boff[i] + C::RING_V + s2);
        else g2l16(kp, uoff[i - LPB], boff[i - LPB] + C::RING_K + s1);
      }
    };
    NHA_FENCE();
    // ---- phase B: value products of unit u on the matrix core, row maximum of unit u+1 on the VALU;
    //      V fragment db is read PD products ahead ----
    float m0 = 0.f, m1 = 0.f;
    auto max_step = [&](int s2) {
      if (s2 == 0 || s2 == 2) {   // to log2 units, relative to the reference
        const int kk = s2 >> 1;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          Sn[kk][r] = fmaf(Sn[kk][r], cs, nm);
          NHA_PIN(Sn[kk][r]);
        }
      }
      if (s2 == 0) m0 = fmaxf(Sn[0][0], Sn[0][1]);
      if (s2 == 1) m1 = fmaxf(Sn[0][2], Sn[0][3]);
      if (s2 == 2) m0 = fmaxf(fmaxf(m0, Sn[1][0]), Sn[1][1]);
      if (s2 == 3) m1 = fmaxf(fmaxf(m1, Sn[1][2]), Sn[1][3]);
      if (s2 == 4) m0 = fmaxf(m0, m1);
      if (s2 == 0 || s2 == 2 || s2 == 4) NHA_PIN(m0);
      if (s2 == 1 || s2 == 3) NHA_PIN(m1);
    };
    bf16x8 vfr[DB];
#pragma unroll
    for (int i = 0; i < PD; ++i) vfr[i] = vfrag(v_c, i);
    Lw = mfma16(ones, Pq, Lw);
    NHA_FENCE();
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if (db + PD < DB) vfr[db + PD] = vfrag(v_c, db + PD);
      O[db] = mfma16(vfr[db], Pq, O[db]);
      if (db % (DB / (2 * LPB)) == 0) request(db / (DB / (2 * LPB)));
      if (db % 3 == 0 && db / 3 < 5) max_step(db / 3);
      NHA_FENCE();
    }
    if (is_edge(u + 1)) {
      mask_unit(Sn, u + 1);
      m0 = max8(Sn);
    }
    // The reference of the window stays where the prologue put it: moving it would mean rescaling 64
    // accumulator registers inside this loop, which costs the loop its registers whether or not the branch
    // is ever taken.  fp32 sums and bf16 probabilities hold 2^BIG above it; a score beyond that sends the
    // wave's 16 rows to the exact pass and is clamped.
    if (__any(m0 > BIG)) {
      if (16 * Q < rows) bad = 1 << Q;   // (a chunk that is not there has no rows)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int r = 0; r < 4; ++r) Sn[kk][r] = fminf(Sn[kk][r], BIG);
    }
    Sc[0] = Sn[0];
    Sc[1] = Sn[1];
    kp -= upr;
    vp -= upr;
    const uint32_t t0 = s0;
    s0 = s1;
    s1 = s2;
    s2 = t0;
  };
  // Most iterations request the next units and nothing else; their scalar instructions are those of two running pointers.
  int u = 0;
#pragma unroll 1
  do {
    step(u, std::false_type{});
    ++u;
    if (u >= 2 * NCH - 2)
#pragma unroll 1
      for (; u + 4 < nunits; ++u) step(u, std::true_type{});
  } while (u + 1 < nunits);
  // ---- the last unit: no further scores; the slot-branch queries are requested meanwhile ----
  {
    const uint32_t v_c = C::RING_V + (u % NR) * UB;
    bf16x8 vf[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) vf[db] = vfrag(v_c, db);
    load_qg();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int r = 0; r < 4; ++r) Sc[kk][r] = fexp2(Sc[kk][r]);
    const bf16x8 Pq = pack_p();
    Lw = mfma16(ones, Pq, Lw);
#pragma unroll
    for (int db = 0; db < DB; ++db) O[db] = mfma16(vf[db], Pq, O[db]);
  }

  // ================= slot branch, folded into the running softmax =================================
  // Every wave its own rows, the waves of both chunks side by side; the next tile is requested when every wave is done with
  // the one before, and what needs no tile is computed while it is on its way.
  // every request of this wave has landed, every wave is done with the rings
  wait_vm<0>();
  lds_barrier();
  if (!early) {
    issue_ta(oT[0][0], 0, 0);
    issue_ta(oT[0][1], 0, 1);
    if (NCH == 2 && second) {
      issue_ta(oT[NCH - 1][0], NCH - 1, 0);
      issue_ta(oT[NCH - 1][1], NCH - 1, 1);
    }
  } else {
    oE2 = C::RING_V + s2, oE2b = C::RING_V + s0;   // (after the loop's last rotation)
  }
  // the window's own log-sum-exp, before the slots join the running softmax
  if (p.lse_swa && kb == 0 && irow < rows) p.lse_swa[(int64_t)(c0 + yrow) * HQ + hq] = (__builtin_amdgcn_logf(Lw[0]) - nm) * LN2;
  take_qg(oE2);
  auto issue_all = [&](auto issue) {
#pragma unroll
    for (int c_ = 0; c_ < NCH; ++c_)
      if (c_ == 0 || second) {
        issue(oT[c_][0], c_, 0);
        issue(oT[c_][1], c_, 1);
      }
  };
  auto landed = [&]() {
    wait_vm<0>();
    lds_barrier();
  };
  if (!early) landed();
  const bool mine = ch == 0 || second;
  const uint32_t t0_ = oT[0][0], t1_ = oT[0][1];
  const uint32_t tile0 = NCH == 2 && ch ? oT[NCH - 1][0] : t0_, tile1 = NCH == 2 && ch ? oT[NCH - 1][1] : t1_;   // halves of the wave's tile
  const uint32_t gco = NCH == 2 && ch ? C::GC2 : C::GC;
  // first table unit of this wave's sub-block (units 0 .. 3 lie in one piece, 4 and 5 in another)
  const uint32_t etab = Q == 3 ? (NCH == 2 && ch ? oE2b : C::ETAB + 4 * 4096) : (NCH == 2 && ch ? oE2 : C::ETAB) + (Q < 2 ? Q : 2) * 4096;
  // E_Q transposed: rows = slots 16 mb + l16, contraction over the tokens 32 pr + {4 kb + e, 16 + 4 kb + e - 4}
  auto etab_tr = [&](int pr, int mb) -> bf16x8 {
    const lbyte* pa = lds + etab + pr * 4096 + (mb >> 1) * 1024 + (mb & 1) * 512 + (uint32_t)((4 * kb + (l16 >> 2)) * 32 + 8 * (l16 & 3));
    struct { s16x4 a, b; } t;
    t.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)pa);
    t.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((NHA_LDS s16x4*)(pa + 2048));
    return __builtin_bit_cast(bf16x8, t);
  };
  // E_Q by rows: row = token 16 jb + l16, contraction over the slots 32 pr + {4 kb + e, 16 + 4 kb + e - 4}
  auto etab_row = [&](int jb, int pr) -> bf16x8 {
    const lbyte* pa = lds + etab + (jb >> 1) * 4096 + (jb & 1) * 2048 + pr * 1024 + l16 * 32 + 8 * kb;
    struct { bf16x4 a, b; } t;
    t.a = *reinterpret_cast<const NHA_LDS bf16x4*>(pa);
    t.b = *reinterpret_cast<const NHA_LDS bf16x4*>(pa + 512);
    return __builtin_bit_cast(bf16x8, t);
  };

  // inter-chunk slot logits: okT[m][i] = sum_d hkT[m][d] q[i][d]
  f32x4 ok[4];
  if (mine) {
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) ok[mb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) ok[mb] = mfma16(kfrag(((mb >> 1) ? tile1 : tile0), mb & 1, ks), qg[ks], ok[mb]);
  }
  // every wave is done with the k-states: the k_gsa rows, and meanwhile the second chunk's tables
  lds_barrier();
  issue_all([&](uint32_t o, int c_, int half) { issue_tb(o, c_, half, t_kg); });
  if (NCH == 2 && second) build_decay_tables(1, C::GC2, oE2, oE2b);
  landed();
  bf16x8 bA[2];
  if (mine) {
    // intra-chunk scores AT[j][i] = sum_d k_gsa[j][d] q[i][d] for row blocks jb <= Q, masked j <= i
    f32x4 at[4];
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) at[jb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        if (jb <= Q) at[jb] = mfma16(kfrag(((jb >> 1) ? tile1 : tile0), jb & 1, ks), qg[ks], at[jb]);
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
      if (jb == Q) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * kb + r > l16) at[jb][r] = 0.f;
      }
    bA[0] = pack8(at[0], at[1]);
    bA[1] = pack8(at[2], at[3]);
  }
  // done with the k_gsa rows: the v-states, and meanwhile the softmax
  lds_barrier();
  issue_all([&](uint32_t o, int c_, int half) { issue_tc(o, c_, half); });
  float psum = 0.f;
  bf16x8 bp[2], bpr[2];   // slot probabilities x exp(gc_i) and x exp(gc_i - gr), B operands
  if (mine) {
    // okT_intra[m][i] = sum_j s_j[m] exp(gr[m] - gc_j[m]) AT[j][i]
    f32x4 oki[4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      oki[mb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int pr = 0; pr < 2; ++pr)
        if (2 * pr <= Q) oki[mb] = mfma16(etab_tr(pr, mb), bA[pr], oki[mb]);
    }
    // combine; the slot logits join the running softmax as one more set of keys
    const int rref = 16 * Q - 1;
    f32x4 egi[4], egr[4];   // exp(gc_i[m]) and exp(gc_i[m] - gr[m]) in accumulator layout
    float xmax = -INFINITY;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const f32x4 gi = *reinterpret_cast<const NHA_LDS f32x4*>(gc_at(gco, irow, 16 * mb + 4 * kb));
      f32x4 gr4 = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (Q > 0) gr4 = *reinterpret_cast<const NHA_LDS f32x4*>(gc_at(gco, rref, 16 * mb + 4 * kb));
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        egi[mb][r] = fexp(gi[r]);
        egr[mb][r] = fexp(gi[r] - gr4[r]);
        ok[mb][r] = (ok[mb][r] * egi[mb][r] + oki[mb][r] * egr[mb][r]) * cs;   // slot logit, log2 units
        xmax = fmaxf(xmax, ok[mb][r]);
      }
    }
    const float ms = max_over_rows(xmax);   // the slots' own maximum
    if (__any(ms + nm > THR)) rescale_acc(fmaxf(ms + nm, 0.f));
    if (p.lse_gsa) {
      float pown = 0.f;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int r = 0; r < 4; ++r) pown += fexp2(ok[mb][r] - ms);
      pown += __shfl_xor(pown, 16, 64);
      pown += __shfl_xor(pown, 32, 64);
      if (kb == 0 && irow < rows) p.lse_gsa[(int64_t)(c0 + yrow) * HQ + hq] = (__builtin_amdgcn_logf(pown) + ms) * LN2;
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ok[mb][r] = fexp2(ok[mb][r] + nm);   // unnormalised slot probabilities
        psum += ok[mb][r];
      }
    psum += __shfl_xor(psum, 16, 64);
    psum += __shfl_xor(psum, 32, 64);
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
      f32x4 x0, x1, y0, y1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x0[r] = ok[2 * pr][r] * egi[2 * pr][r];
        x1[r] = ok[2 * pr + 1][r] * egi[2 * pr + 1][r];
        y0[r] = ok[2 * pr][r] * egr[2 * pr][r];
        y1[r] = ok[2 * pr + 1][r] * egr[2 * pr + 1][r];
      }
      bp[pr] = pack8(x0, x1);
      bpr[pr] = pack8(y0, y1);
    }
  }
  landed();
  // slot read, inter-chunk part: O^T[d][i] += sum_m hv[m][d] (p[i][m] exp(gc_i[m]))
  if (mine) {
#pragma unroll
    for (int pr = 0; pr < 2; ++pr)
#pragma unroll
      for (int db = 0; db < DB; ++db) O[db] = mfma16(vfrag((pr ? tile1 : tile0), db), bp[pr], O[db]);
  }
  // done with the v-states: the v rows, and meanwhile their weights
  lds_barrier();
  issue_all([&](uint32_t o, int c_, int half) { issue_tb(o, c_, half, vbase); });
  bf16x8 bAv[2];
  if (mine) {
    // intra-chunk part: AvT[j][i] = sum_m s_j[m] exp(gr[m]-gc_j[m]) (p[i][m] exp(gc_i[m]-gr[m])), j <= i
    f32x4 av[4];
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) {
      av[jb] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (jb <= Q) {
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) av[jb] = mfma16(etab_row(jb, pr), bpr[pr], av[jb]);
        if (jb == Q) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (4 * kb + r > l16) av[jb][r] = 0.f;
        }
      }
    }
    bAv[0] = pack8(av[0], av[1]);
    bAv[1] = pack8(av[2], av[3]);
  }
  landed();
  if (mine) {
#pragma unroll
    for (int pr = 0; pr < 2; ++pr)
      if (2 * pr <= Q) {
#pragma unroll
        for (int db = 0; db < DB; ++db) O[db] = mfma16(vfrag((pr ? tile1 : tile0), db), bAv[pr], O[db]);
      }
  }

  // ---- epilogue: 16-byte stores (the lanes of an even 16-lane row keep block db, those of the odd
  //      row block db + 1, and the two trade their halves) -------------------------------------------
  {
    const float inv = 1.f / (Lw[0] + psum);
    bf16_t* op = p.o + ((int64_t)(c0 + yrow) * HQ + hq) * D;
#pragma unroll
    for (int db = 0; db < DB; db += 2) {
      unsigned a[2], b[2];
      a[0] = cvt2(O[db][0] * inv, O[db][1] * inv);
      a[1] = cvt2(O[db][2] * inv, O[db][3] * inv);
      b[0] = cvt2(O[db + 1][0] * inv, O[db + 1][1] * inv);
      b[1] = cvt2(O[db + 1][2] * inv, O[db + 1][3] * inv);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const auto sw = __builtin_amdgcn_permlane16_swap(a[e], b[e], false, false);
        a[e] = sw[0];
        b[e] = sw[1];
      }
      const int dcol = 16 * (db + (kb & 1)) + 8 * (kb >> 1);
      if (irow < rows) *reinterpret_cast<uint4*>(op + dcol) = make_uint4(a[0], a[1], b[0], b[1]);
    }
  }
  // ---- rows that have to be formed again (prefill_exact.h) ------------------------------------------
  lds_barrier();
  if (lane == 0) *reinterpret_cast<NHA_LDS int*>(lds + 4 * wave) = bad;
  lds_barrier();
#pragma unroll
  for (int w = 0; w < NW; ++w) exact[w >> 2] |= *reinterpret_cast<const NHA_LDS int*>(lds + 4 * w);
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int bits = __builtin_amdgcn_readfirstlane(exact[c]);
    if (bits == 0) continue;
    before_exact();
    exact_rows<D, NCH>(arguments_again(), reinterpret_cast<float*>(smem_), chunk + c, h, hq, 1, bits);
  }
}

}  // namespace

// Served: K == V == 256 with any grouping of query heads (each head walks its kv-head's window on its
// own).  The per-lane byte offsets of the LDS-direct loads are 32 bits: the tensors of one call must
// stay below 4 GiB.
bool prefill_ring256_supported(const mf::MP& p, int D) {
  if (D != 256) return false;
  return (int64_t)p.T_tot * p.H * D * 2 < ((int64_t)1 << 32) && (int64_t)p.T_tot * p.H * MS * 2 < ((int64_t)1 << 32);
}

namespace {
template <int NCH>
int launch_ring256(const mf::MP& p, hipStream_t st) {
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute((const void*)ring256_out_kernel<NCH>, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg<NCH>::BYTES); });
  if (attr_err != hipSuccess) {
    set_error("nha_prefill_fwd(mfma): cannot reserve %d bytes of LDS: %s", Cfg<NCH>::BYTES, hipGetErrorString(attr_err));
    return NHA_ERR_LAUNCH;
  }
  hipLaunchKernelGGL((ring256_out_kernel<NCH>), NCH == 1 ? dim3(p.HQ, p.NT) : pair_grid(p.HQ, p.NT, p.N), dim3(256 * NCH), Cfg<NCH>::BYTES, st, p);
  NHA_CHECK_LAUNCH("nha_prefill_fwd(mfma output pass, ring, head size 256)");
  return NHA_OK;
}
}  // namespace

int prefill_ring256_launch(const mf::MP& p, hipStream_t st) {
  // two chunks per workgroup unless most sequences have a single chunk (fewer than three chunks per two sequences):
  // there the second half of a two-chunk workgroup would mostly idle
  const bool one = 2 * (int64_t)p.NT < 3 * (int64_t)p.N;
  return one ? launch_ring256<1>(p, st) : launch_ring256<2>(p, st);
}

}  // namespace nha
