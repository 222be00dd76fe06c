// Window branch of the NHA prefill backward for K == V == 256 (bf16): the streams of prefill_bwd_ring.hip, cut for a head size
// at which neither the rows of a wave beside its sums nor both gradients fit one wave's registers.  Two waves, one of each
// kind, share 32 rows on one SIMD:
//
// ring256_dq_kernel: one workgroup of 8 waves = two 64-token chunks of one query head, four pairs of waves with 32 queries
//   each.  The window's K / V rows stream through a ring in units of 32 keys; wave r of a pair forms S^T, dP^T and dS^T of
//   the unit's 16-key half r, the halves meet in LDS as bf16 operands, and a unit later the wave adds its 128 of the 256
//   columns of dQ^T += K^T dS^T.  A fragment read from LDS feeds two products (one in bwd_dq_kernel: 16 queries a wave).
// ring256_dkv_kernel: one workgroup of 8 waves = 128 keys of one kv-head, four pairs of waves with 32 keys each; the q / do
//   rows of every query head of the group stream in items of 32 queries.  Wave 0 of a pair has K rows and dV: S = Q K^T,
//   P, dV^T += dO^T P; wave 1 has V rows and dK, one item behind: dP = dO V^T, dS from P as the other left it in LDS in
//   fp32, dK^T += Q^T dS.  (bwd_dkv_kernel forms S twice, once per gradient.)
//
// Products of one kind of wave fill the other's exponentials and waits.  Bound: LDS reads and matrix instructions side by side in the
// stream, and the first 128 KB of a workgroup, with nothing else on the CU.  B=8, T=2048, 4 heads, W = 512 (bwd_dq_kernel and
// bwd_dkv_kernel / these): dq 98 / 88 us, dk and dv 190 / 132.
#include "common.h"
#include "mfma_common.h"

#include <mutex>

namespace nha {
namespace {
using namespace mf;

constexpr int D = 256, KS = D / 32, DB = D / 16;
constexpr int UB = 32 * D * 2;        // a 32-row tile (LineTile)
constexpr int ROWS = 128;             // rows (queries or keys) of a workgroup

struct WinP {
  const bf16_t *q, *k, *v, *dout;          // q_swa [T,HQ,D]; k_swa, v [T,H,D]; dout [T,HQ,D]
  const float *lse_swa, *lse_gsa, *delta;  // [T,HQ]
  float2* ld;                              // [T,HQ] (-lse log2(e), -delta): left by the dq kernel, read by the other
  const float* dvs;                        // [T,H,D] slot-branch part of dv
  float *wk, *wv;                          // fp32 sums of the dk / dv kernel's parts, [gridDim.z][T,H,D] (pd floats each)
  int64_t pd;
  bf16_t *dq, *dk, *dv;
  const int32_t *cu, *coff;
  int HQ, H, NG, N, wl;
  float scale;
};

#define FENCE __builtin_amdgcn_sched_barrier(0)

// The workgroup's 128 rows of a [*, heads, D] tensor into LDS as four tiles of 32 rows from byte address `at` on, by all waves (eight
// loads each): a wave's own fragments loaded from global memory are 16-byte pieces of 16 rows, the slowest pattern there is
// (LineTile), and came twice, for both waves of a pair.  Rows past the end repeat row `last`.
__device__ __forceinline__ void load_rows(const bf16_t* src, int64_t stride, int first, int last, uint32_t at, int wave, int lane) {
  const uint32_t col = LineTile<D>::load_col(wave, lane);
#pragma unroll
  for (int i = 0; i < ROWS / 16; ++i) {
    int r = 16 * i + LineTile<D>::load_row(lane);
    r = first + r < last ? r : last - first;
    g2l16(src + (int64_t)first * stride, ((uint32_t)r * (uint32_t)stride + col) * 2,
          at + wave * 1024 + (i >> 1) * UB + (i & 1) * LineTile<D>::HALF);
  }
}

constexpr int DQ_NR = 4;                          // ring slots
constexpr int DQ_UNIT = 2 * UB;                   // K tile | V tile
constexpr int DQ_LPW = 4;                         // LDS-direct loads per wave and unit (32 blocks, 8 waves)
constexpr int DQ_EX = DQ_NR * DQ_UNIT;            // dS halves: [unit parity][pair][half][16-query block][lane] 8 bytes
constexpr int DQ_BYTES = DQ_EX + 2 * 8 * 1024;

__global__ __launch_bounds__(512, 1) void ring256_dq_kernel(const WinP p) {
  extern __shared__ __align__(1024) unsigned char smem_[];
  lbyte* const lds = (lbyte*)smem_;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kb = lane >> 4, pair = wave & 3, half = wave >> 2;
  const int H = p.H, HQ = p.HQ;
  int hq, n, it;
  if (!pair_tile(p.coff, p.N, HQ, p.NG, hq, n, it)) return;
  const int h = hq / p.NG;
  const int bos = p.cu[n], eos = p.cu[n + 1], c0 = bos + it * BT;
  const int rows = (eos - c0) < ROWS ? (eos - c0) : ROWS;
  const int row0 = 32 * pair;   // first query of the wave, relative to c0
  const float cs = p.scale * LOG2E;

  // unit u covers keys [top - 32 u - 32, top - 32 u): from the workgroup's last rows down; top - bos is a multiple of 32, so no
  // unit starts before its sequence; rows past eos (unit 0 only) are read from row eos - 1: masked, finite
  const int top = c0 + ((rows + 31) & ~31);
  int lowest = bos;
  if (p.wl >= 0 && c0 - p.wl > bos) lowest = c0 - p.wl;
  const int nunits = (top - lowest + 31) / 32;
  const bf16_t* const kbase = p.k + ((int64_t)bos * H + h) * D;
  const bf16_t* const vbase = p.v + ((int64_t)bos * H + h) * D;
  auto issue_unit = [&](int u) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    // a wave loads 32 columns of both tiles
    const uint32_t dst = lds0 + (u & (DQ_NR - 1)) * DQ_UNIT + wave * 1024, pcol = LineTile<D>::load_col(wave, lane);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      int r = top - 32 * (u + 1) + 16 * i + LineTile<D>::load_row(lane);
      r = r < eos ? r : eos - 1;
      const uint32_t off = ((uint32_t)(r - bos) * (uint32_t)(H * D) + pcol) * 2;
      g2l16(kbase, off, dst + i * LineTile<D>::HALF);
      g2l16(vbase, off, dst + UB + i * LineTile<D>::HALF);
    }
  };
  // q and do rows through the ring's slots: q where the first two units go, do where the next two go
  load_rows(p.q + (int64_t)hq * D, (int64_t)HQ * D, c0, eos - 1, lds0, wave, lane);
  load_rows(p.dout + (int64_t)hq * D, (int64_t)HQ * D, c0, eos - 1, lds0 + 2 * DQ_UNIT, wave, lane);
  float nlse[2], ndl[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int y = row0 + 16 * qb + l16;
    const bool valid = y < rows;
    const int64_t tq = (int64_t)(c0 + (valid ? y : 0)) * HQ + hq;
    const float ls = p.lse_swa[tq], lg = p.lse_gsa[tq], mx = fmaxf(ls, lg);
    nlse[qb] = valid ? -(mx + logf(expf(ls - mx) + expf(lg - mx))) * LOG2E : -INFINITY;   // rows past the end weigh nothing
    ndl[qb] = -p.delta[tq];
    if (valid && half == 0 && kb == 0) p.ld[tq] = make_float2(nlse[qb], ndl[qb]);
    // in their registers before the loop: the compiler's wait for them inside it would drain the LDS-direct loads as well
    asm volatile("" : "+v"(nlse[qb]));
    asm volatile("" : "+v"(ndl[qb]));
  }
  bf16x8 qf[2][KS], df[2][KS];
  {
    const LineTile<D> rd(lds, lane);
    wait_vm<0>();
    lds_barrier();
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[qb][ks] = rd.row(pair * UB, qb, ks);
    lds_barrier();   // (waits for this wave's reads)
    issue_unit(0);
    if (nunits > 1) issue_unit(1);
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) df[qb][ks] = rd.row(2 * DQ_UNIT + pair * UB, qb, ks);
  }
  f32x4 dQ[DB / 2][2];
#pragma unroll
  for (int db = 0; db < DB / 2; ++db) dQ[db][0] = dQ[db][1] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // no query of the pair sees a key of unit u
  auto no_work = [&](int u) {
    const int x0 = top - c0 - 32 * (u + 1);
    return row0 >= rows || x0 > row0 + 31 || (p.wl >= 0 && x0 + 31 < row0 - p.wl);
  };
  for (int t = 0; t <= nunits; ++t) {
    // unit t has landed (this wave's part), then everybody's, and the dS of unit t - 1 too; unit t + 1 stays in flight
    if (t + 1 < nunits) wait_vm<DQ_LPW>();
    else wait_vm<0>();
    lds_barrier();
    if (t + 2 < nunits) issue_unit(t + 2);   // the slot of unit t - 2
    const bool now = t < nunits && !no_work(t), before = t > 0 && !no_work(t - 1);
    const uint32_t base = (uint32_t)((t & (DQ_NR - 1)) * DQ_UNIT);
    int lc = threadIdx.x & 63;
    asm volatile("" : "+v"(lc));   // what follows from the lane's number is derived anew: there are no registers to keep it
    const LineTile<D> rd(lds, lc);
    const int l16 = lc & 15, kb = lc >> 4;
    lbyte* const ex = lds + DQ_EX + pair * 2048 + lc * 8;   // + 8192 (unit parity) + 1024 (half) + 512 (16-query block)
    f32x4 S[2], dP[2];
    if (now) {
      bf16x8 ka[KS], va[KS];
      ka[0] = rd.row(base, half, 0);
      ka[1] = rd.row(base, half, 1);
      S[0] = S[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        FENCE;
        if (ks + 2 < KS) ka[ks + 2] = rd.row(base, half, ks + 2);
        else va[ks + 2 - KS] = rd.row(base + UB, half, ks + 2 - KS);
        FENCE;
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) S[qb] = mfma16(ka[ks], qf[qb][ks], S[qb]);
      }
      FENCE;
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[qb][r] = S[qb][r] * cs + nlse[qb];
      const int x0 = top - c0 - 32 * (t + 1);
      if (x0 + 31 > row0 || (p.wl >= 0 && x0 < row0 + 31 - p.wl)) {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int x = x0 + 16 * half + 4 * kb + r, y = row0 + 16 * qb + l16;
            const bool ok = (x <= y) && (p.wl < 0 || x >= y - p.wl);
            if (!ok) S[qb][r] = -INFINITY;
          }
      }
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) dP[qb] = (f32x4){ndl[qb], ndl[qb], ndl[qb], ndl[qb]};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        FENCE;
        if (ks + 2 < KS) va[ks + 2] = rd.row(base + UB, half, ks + 2);
        FENCE;
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) dP[qb] = mfma16(va[ks], df[qb][ks], dP[qb]);
        S[ks >> 2][ks & 3] = fexp2(S[ks >> 2][ks & 3]);
      }
      FENCE;
    }
    auto leave_ds = [&](int qb) {
      bf16x4 x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = (__bf16)(S[qb][r] * dP[qb][r]);
      *reinterpret_cast<NHA_LDS bf16x4*>(ex + (t & 1) * 8192 + half * 1024 + qb * 512) = x;
    };
    if (before) {
      const uint32_t kt = (uint32_t)(((t - 1) & (DQ_NR - 1)) * DQ_UNIT);
      bf16x8 ds[2], kf[DB / 2];
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        struct { bf16x4 a, b; } x;
        const lbyte* const at = ex + ((t - 1) & 1) * 8192 + qb * 512;
        x.a = *reinterpret_cast<const NHA_LDS bf16x4*>(at);
        x.b = *reinterpret_cast<const NHA_LDS bf16x4*>(at + 1024);
        ds[qb] = __builtin_bit_cast(bf16x8, x);
      }
      kf[0] = rd.col(kt, half * (DB / 2));
      kf[1] = rd.col(kt, half * (DB / 2) + 1);
#pragma unroll
      for (int db = 0; db < DB / 2; ++db) {
        FENCE;
        if (db + 2 < DB / 2) kf[db + 2] = rd.col(kt, half * (DB / 2) + db + 2);
        FENCE;
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) dQ[db][qb] = mfma16(kf[db], ds[qb], dQ[db][qb]);
        if (now && (db == 1 || db == 2)) leave_ds(db - 1);
      }
      FENCE;
    } else if (now) {
      leave_ds(0);
      leave_ds(1);
    }
  }
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int y = row0 + 16 * qb + l16;
    if (y >= rows) continue;
    bf16_t* const op = p.dq + ((int64_t)(c0 + y) * HQ + hq) * D + half * (D / 2) + 4 * kb;
#pragma unroll
    for (int db = 0; db < DB / 2; ++db) {
      bf16x4 pk;
#pragma unroll
      for (int r = 0; r < 4; ++r) pk[r] = (__bf16)(dQ[db][qb][r] * p.scale);
      *reinterpret_cast<bf16x4*>(op + 16 * db) = pk;
    }
  }
}

// ------------------------------------------------------------------------------------------------------
constexpr int KV_NR = 3;                          // ring slots
constexpr int KV_Q = 0, KV_O = UB, KV_LD = 2 * UB, KV_ITEM = 2 * UB + 256;   // q tile | do tile | 32 (lse, delta) pairs
constexpr int KV_LPW = 4;                         // tile loads per wave and item
constexpr int KV_P = KV_NR * KV_ITEM;             // P in fp32: [item parity][pair][quad][lane] 16 bytes
constexpr int KV_BYTES = KV_P + 2 * 4 * 4096;
constexpr int UPG = ROWS / 32;                    // 32-query units that a key group spans

// PARTS: a kv-head's query heads are shared out over gridDim.z, and fp32 sums take the place of dk and dv
template <bool PARTS>
__global__ __launch_bounds__(512, 1) void ring256_dkv_kernel(const WinP p) {
  extern __shared__ __align__(1024) unsigned char smem_[];
  lbyte* const lds = (lbyte*)smem_;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kb = lane >> 4, pair = wave & 3;
  const bool second = wave >= 4;   // the wave with V rows and dK, an item behind
  const int H = p.H, HQ = p.HQ, NG = p.NG;
  int h, n, it;
  if (!pair_tile(p.coff, p.N, H, 1, h, n, it)) return;
  const int hq0 = PARTS ? (h * gridDim.z + blockIdx.z) * NG : h * NG;
  const int bos = p.cu[n], eos = p.cu[n + 1], c0 = bos + it * BT;
  const int rows = (eos - c0) < ROWS ? (eos - c0) : ROWS;
  const int row0 = 32 * pair;   // first key of the wave, relative to c0
  const float cs = p.scale * LOG2E;
  // queries that see a key of the workgroup: [c0, qend), in items of 32 per query head
  int qend = eos;
  if (p.wl >= 0 && c0 + rows + p.wl < eos) qend = c0 + rows + p.wl;
  const int nun = (qend - c0 + 31) / 32;   // >= 1
  const int total = NG * nun;
  // Neighbouring key groups of a sequence run at the same time on one XCD: each walks the units of a head cyclically from where
  // the walk of the sequence's first group is by then, so that a row is requested by all of them at about the same time.
  const int rot = (nun - (UPG * (it >> 1)) % nun) % nun;
  struct Walk { int g, u, left; };
  auto advance = [&](Walk& w) {
    w.u = w.u + 1 == nun ? 0 : w.u + 1;
    if (--w.left == 0) {
      w.left = nun;
      w.u = rot;
      ++w.g;
    }
  };
  Walk iw = {0, rot, nun};
  int islot = 0;
  auto issue_item = [&]() {   // rows past eos are read from row eos - 1: masked, finite
    int ln = threadIdx.x & 63;
    asm volatile("" : "+v"(ln));   // derived anew at every request: kept across the loop it would cost registers
    const int hq = hq0 + iw.g, q0 = c0 + 32 * iw.u;
    const bf16_t* const qbase = p.q + ((int64_t)bos * HQ + hq) * D;
    const bf16_t* const obase = p.dout + ((int64_t)bos * HQ + hq) * D;
    const uint32_t dst = lds0 + islot * KV_ITEM + wave * 1024, pcol = LineTile<D>::load_col(wave, ln);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      int r = q0 + 16 * i + LineTile<D>::load_row(ln);
      r = r < eos ? r : eos - 1;
      const uint32_t off = ((uint32_t)(r - bos) * (uint32_t)(HQ * D) + pcol) * 2;
      g2l16(qbase, off, dst + KV_Q + i * LineTile<D>::HALF);
      g2l16(obase, off, dst + KV_O + i * LineTile<D>::HALF);
    }
    if (wave == 0) {
      int r = q0 + (ln >> 1);
      r = r < eos ? r : eos - 1;
      g2l4(p.ld, (uint32_t)(((int64_t)r * HQ + hq) * 2 + (ln & 1)) * 4u, lds0 + islot * KV_ITEM + KV_LD);
    }
    advance(iw);
    islot = islot + 1 == KV_NR ? 0 : islot + 1;
  };
  // K or V rows of this lane's keys, one per 16-key block, through the room of the ring
  static_assert(2 * 4 * UB <= KV_BYTES, "K and V rows of the workgroup fit the LDS");
  load_rows(p.k + (int64_t)h * D, (int64_t)H * D, c0, eos - 1, lds0, wave, lane);
  load_rows(p.v + (int64_t)h * D, (int64_t)H * D, c0, eos - 1, lds0 + 4 * UB, wave, lane);
  bf16x8 own[2][KS];
  {
    const LineTile<D> rd(lds, lane);
    wait_vm<0>();
    lds_barrier();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) own[kk][ks] = rd.row((second ? 4 * UB : 0) + pair * UB, kk, ks);
    lds_barrier();   // (waits for this wave's reads)
  }
  int issued = 0;
  for (; issued < KV_NR && issued < total; ++issued) issue_item();
  f32x4 acc[DB][2];   // dV^T or dK^T
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db][0] = acc[db][1] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // no query of unit u sees a key of the pair
  auto no_work = [&](int u) { return row0 >= rows || 32 * u + 31 < row0 || (p.wl >= 0 && 32 * u > row0 + 31 + p.wl); };
  Walk w = {0, rot, nun};   // this wave's item
  int slot = 0;
  for (int t = 0; t <= total; ++t) {
    // item t has landed (this wave's part; wave 0 carries one load more), then everybody's, and P of item t - 1 too
    const int younger = issued - (t + 1);
    if (younger >= 2) {
      if (wave == 0) wait_vm<2 * (KV_LPW + 1)>();
      else wait_vm<2 * KV_LPW>();
    } else if (younger == 1) {
      if (wave == 0) wait_vm<KV_LPW + 1>();
      else wait_vm<KV_LPW>();
    } else {
      wait_vm<0>();
    }
    lds_barrier();
    if (t >= 2 && issued < total) {   // into the slot of item t - 2
      issue_item();
      ++issued;
    }
    const bool mine = second ? t > 0 : t < total;
    const int u = w.u;
    const uint32_t base = (uint32_t)(slot * KV_ITEM);
    if (mine) {
      advance(w);
      slot = slot + 1 == KV_NR ? 0 : slot + 1;
    }
    if (mine && !no_work(u)) {
      int lc = threadIdx.x & 63;
      asm volatile("" : "+v"(lc));
      const LineTile<D> rd(lds, lc);
      const int kb = lc >> 4;
      const uint32_t rt = base + (second ? KV_O : KV_Q), tt = base + (second ? KV_Q : KV_O);
      lbyte* const pb = lds + KV_P + (second ? (t + 1) & 1 : t & 1) * 16384 + pair * 4096 + lc * 16;
      // scores (16-query block q & 1, 16-key block q >> 1): rows of the accumulators are the queries 16 qb + 4 kb + r, the column is
      // this lane's key of its block
      // (-lse, -delta) of rows 16 qb + 4 kb + r: -delta is where dP starts from
      auto pairs = [&](int qb) {
        const NHA_LDS f32x4* lp = reinterpret_cast<const NHA_LDS f32x4*>(lds + base + KV_LD + (16 * qb + 4 * kb) * 8);
        const f32x4 a0 = lp[0], a1 = lp[1];
        return second ? (f32x4){a0[1], a0[3], a1[1], a1[3]} : (f32x4){a0[0], a0[2], a1[0], a1[2]};
      };
      f32x4 C[4];
      bf16x8 x[KS][2], y[DB], B[2];
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        x[0][qb] = rd.row(rt, qb, 0);
        C[qb] = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (second) C[qb] = pairs(qb);
        C[qb + 2] = C[qb];
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        FENCE;
        if (ks + 1 < KS) {
          x[ks + 1][0] = rd.row(rt, 0, ks + 1);
          x[ks + 1][1] = rd.row(rt, 1, ks + 1);
        } else {
          y[0] = rd.col(tt, 0);
        }
        FENCE;
#pragma unroll
        for (int q = 0; q < 4; ++q) C[q] = mfma16(x[ks][q & 1], own[q >> 1][ks], C[q]);
      }
      FENCE;
      if (second) {
#pragma unroll
        for (int q = 0; q < 4; ++q) C[q] *= *reinterpret_cast<const NHA_LDS f32x4*>(pb + q * 1024);
      } else {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          const f32x4 nl = pairs(qb);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            C[qb][r] = C[qb][r] * cs + nl[r];
            C[qb + 2][r] = C[qb + 2][r] * cs + nl[r];
          }
        }
        if (32 * u < row0 + 31 || (p.wl >= 0 && 32 * u + 31 > row0 + p.wl) || c0 + 32 * u + 32 > eos) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int yq = 32 * u + 16 * (q & 1) + 4 * kb + r, xk = row0 + 16 * (q >> 1) + (lc & 15);
              const bool ok = (xk <= yq) && (p.wl < 0 || yq - xk <= p.wl) && (c0 + yq < eos);
              if (!ok) C[q][r] = -INFINITY;
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int r = 0; r < 4; ++r) C[q][r] = fexp2(C[q][r]);
          *reinterpret_cast<NHA_LDS f32x4*>(pb + q * 1024) = C[q];
        }
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) B[kk] = pack8(C[2 * kk], C[2 * kk + 1]);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        FENCE;
        if (db + 1 < DB) y[db + 1] = rd.col(tt, db + 1);
        FENCE;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) acc[db][kk] = mfma16(y[db], B[kk], acc[db][kk]);
      }
      FENCE;
    }
  }
  int le = threadIdx.x & 63;
  asm volatile("" : "+v"(le));
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int x = row0 + 16 * kk + (le & 15);
    if (x >= rows) continue;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int64_t off = ((int64_t)(c0 + x) * H + h) * D + 16 * db + 4 * (le >> 4);
      if constexpr (PARTS) {
        *reinterpret_cast<f32x4*>((second ? p.wk : p.wv) + blockIdx.z * p.pd + off) = second ? acc[db][kk] * p.scale : acc[db][kk];
        continue;
      }
      bf16x4 pk;
      if (second) {
#pragma unroll
        for (int r = 0; r < 4; ++r) pk[r] = (__bf16)(acc[db][kk][r] * p.scale);
        *reinterpret_cast<bf16x4*>(p.dk + off) = pk;
      } else {
        const float4 sv = *reinterpret_cast<const float4*>(p.dvs + off);
        pk[0] = (__bf16)(acc[db][kk][0] + sv.x);
        pk[1] = (__bf16)(acc[db][kk][1] + sv.y);
        pk[2] = (__bf16)(acc[db][kk][2] + sv.z);
        pk[3] = (__bf16)(acc[db][kk][3] + sv.w);
        *reinterpret_cast<bf16x4*>(p.dv + off) = pk;
      }
    }
  }
}

WinP make_p(const NhaPrefillBwdArgs* a, const float* delta, float2* ld, const float* dvs) {
  WinP p;
  p.q = (const bf16_t*)a->q_swa; p.k = (const bf16_t*)a->k_swa; p.v = (const bf16_t*)a->v; p.dout = (const bf16_t*)a->dout;
  p.lse_swa = a->lse_swa; p.lse_gsa = a->lse_gsa; p.delta = delta; p.ld = ld; p.dvs = dvs;
  p.dq = (bf16_t*)a->dq_swa; p.dk = (bf16_t*)a->dk_swa; p.dv = (bf16_t*)a->dv;
  p.wk = p.wv = nullptr; p.pd = 0;
  p.cu = a->cu_seqlens; p.coff = a->chunk_offsets;
  p.HQ = a->HQ; p.H = a->H; p.NG = a->HQ / a->H; p.N = a->N; p.wl = a->wl; p.scale = a->scale;
  return p;
}

template <class K>
int launch(K kernel, int lds, int heads, int parts, const NhaPrefillBwdArgs* a, const WinP& p, std::once_flag& once, hipError_t& err, const char* what) {
  std::call_once(once, [&] { err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds); });
  if (err != hipSuccess) {
    set_error("nha_prefill_bwd: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(err));
    return NHA_ERR_LAUNCH;
  }
  dim3 grid = pair_grid(heads, a->NT, a->N);
  grid.z = parts;
  hipLaunchKernelGGL(kernel, grid, dim3(512), lds, (hipStream_t)a->stream, p);
  NHA_CHECK_LAUNCH(what);
  return NHA_OK;
}

}  // namespace

// tensors of one call below 4 GiB: 32-bit lane offsets of the LDS-direct loads
static bool served(const NhaPrefillBwdArgs* a) {
  return a->K == 256 && a->V == 256 && (int64_t)a->T_tot * a->HQ * 256 * 2 < ((int64_t)1 << 32);
}

// A sequence with an odd number of chunks leaves half of its last workgroup of 128 rows empty, which calls of short sequences feel.
// Whether `percent` of the halves have rows: equally long sequences are taken as such (c of 2 ceil(c / 2) halves at c chunks each);
// of others, the shorter ones weighing more than their rows, three in four as odd.
static bool filled(const NhaPrefillBwdArgs* a, int percent) {
  const int64_t NT = a->NT, N = a->N;
  const int64_t halves = NT % N == 0 ? 2 * N * ((NT / N + 1) / 2) : NT + 3 * N / 4;
  return 100 * NT >= percent * halves;
}

// A workgroup of 128 rows begins with 128 KB that nothing hides (11 of bwd_dq_kernel's 64 rows wait on a CU shared by two), which
// long windows pay back.  us, bwd_dq_kernel / ring256_dq_kernel, 4 heads: W = 64 13.3 / 17.7 at 1000 tokens and 49 / 52 at 3 x
// 5000; W = 256 23 / 26 at 1000 and 129 / 128 at 30000 packed; W = 512 35.0 / 35.2 at 1000, 38 / 38 at 4000, 52 / 45 at 2 x 4000,
// 98 / 88 at 3 x 5000; W = 1024 56 / 50 at 1000, 80 / 66 at 2 x 4000.
// Short sequences, W = 512: 120 of 130 tokens (75 % filled) 54 / 74, of 256 (100 %) 116 / 102, of 400 (88 %) 175 / 223, of 513 (90
// %) 269 / 270, 8 of 700 (92 %) 46 / 37, 60 of 960 (94 %) 264 / 265; ragged, 500 of 300 on average (87 %) 500 / 570, 80 of 400 (90
// %) 142 / 145, 60 of 600 (93 %) 160 / 157.
bool bwd_ring256_dq_supported(const NhaPrefillBwdArgs* a) { return served(a) && (a->wl < 0 || a->wl >= 384) && filled(a, 91); }

// Parts of a kv-head's query heads: as many as all workgroups still have a place at once in, windows of 192 keys or more.  8 / 2
// heads, bwd_dkv_kernel / ring256_dkv_kernel in parts and their sum, us: 5500 tokens, W = 900 (2 parts) 247 / 142, 2 x 3000, W = 300
// 107 / 76, 2786, W = 254 52 / 44, 4000, W = 512 91 / 65; 1500 packed, W = 700 (4) 73 / 44; short windows 4000, W = 64 29 / 38, 2500, W
// = 64 28 / 32, 700, W = 100 36 / 32.
int bwd_ring256_dkv_parts(const NhaPrefillBwdArgs* a) {
  if (!served(a) || (a->wl >= 0 && a->wl < 192)) return 1;
  const int NG = a->HQ / a->H;
  const int64_t groups = (int64_t)a->H * ((a->NT + a->N) / 2);
  int parts = 1;
  while (parts < 8 && NG % (2 * parts) == 0 && 2 * parts * groups <= 256) parts *= 2;
  return parts;
}

// One workgroup of 128 keys fills a CU where bwd_dkv_kernel has four of 64 (two per CU), and walks all heads of its group: it pays
// from half of the chip on, and with one head and short windows not yet.  us, bwd_dkv_kernel / ring256_dkv_kernel: 4 / 4 heads, 2 x
// 4000 tokens (256 groups) W = 64 47 / 43, W = 256 69 / 52, W = 512 102 / 73, W = 1024 149 / 92; 2 x 6000 (376) 72 / 81, 104 / 101,
// -, 235 / 178; 4000 tokens (128) 25 / 33, 36 / 43, 52 / 60, 82 / 83; 8 / 2 heads, 2 x 4000 (128) 50 / 69, 95 / 110, 153 / 178, 262
// / 264; 2 x 6000 (188) 86 / 74, 172 / 115, -, 506 / 270.
// Short sequences: 4 / 4 heads, W = 512, 120 of 130 tokens 105 / 142, of 256 211 / 170, of 400 347 / 382, of 513 523 / 435; ragged,
// 240 of 150 on average (79 % filled) 229 / 251, 160 of 200 (83 %) 217 / 215, 80 of 400 (90 %) 260 / 231.  8 / 2 heads, W = 512:
// 1000 of 130 836 / 1030, 120 of 300 (83 %) 331 / 266; ragged, 300 of 100 (73 %) 212 / 214, 240 of 150 306 / 257.  8 / 2 heads, W =
// 64: 120 of 130 122 / 130, of 256 198 / 157, of 400 297 / 302, of 600 443 / 375; ragged, 300 of 100 194 / 216, 80 of 400 201 /
// 217, 500 of 600 (93 %) 1807 / 1525.
bool bwd_ring256_dkv_supported(const NhaPrefillBwdArgs* a) {
  if (!served(a) || ((int64_t)a->H * a->NT <= 256 && bwd_ring256_dkv_parts(a) == 1)) return false;
  const bool wide = a->wl < 0 || a->wl >= 192;
  if (a->HQ > a->H) return filled(a, wide ? 78 : 91);
  return wide && filled(a, 88);
}

int bwd_ring256_dq(const NhaPrefillBwdArgs* a, const float* delta, float2* ld) {
  static std::once_flag once;
  static hipError_t err = hipSuccess;
  return launch(ring256_dq_kernel, DQ_BYTES, a->HQ, 1, a, make_p(a, delta, ld, nullptr), once, err, "nha_prefill_bwd(window dq, ring 256)");
}

int bwd_ring256_dkv(const NhaPrefillBwdArgs* a, const float2* ld, const float* dvs, int parts, float* wk, float* wv) {
  static std::once_flag once, once_parts;
  static hipError_t err = hipSuccess, err_parts = hipSuccess;
  WinP p = make_p(a, nullptr, (float2*)ld, dvs);
  p.wk = wk; p.wv = wv; p.pd = (int64_t)a->T_tot * a->H * a->K;
  p.NG /= parts;
  const char* const what = "nha_prefill_bwd(window dk, dv, ring 256)";
  if (parts > 1) return launch(ring256_dkv_kernel<true>, KV_BYTES, a->H, parts, a, p, once_parts, err_parts, what);
  return launch(ring256_dkv_kernel<false>, KV_BYTES, a->H, 1, a, p, once, err, what);
}

}  // namespace nha
