// Slot branch of the NHA prefill backward on the matrix cores of gfx950 (bf16, K == V == D in {64,128,256}, M == 64):
// everything of a chunk that does not involve the state gradient carried in from later chunks, in ONE launch, one
// workgroup per (chunk, kv-head) that walks the query heads of the group (nha_fla/ops/nha/chunk_gsa.py:52-122; the
// quantities are those of prefill_bwd.hip).  Per head, with rows i, j, r of the chunk, slots m, k' / v' / s read at the
// source token of their row, and ref_b the gate cumsum at the start of a 32-row half (ref_0 = 0, ref_1 = gc_31):
//   A = q k'^T, B = do v'^T (j <= i), U = q hk0^T, P0 = do hv0^T, delta = do . o
//   Y = s o e^(ref - gc);   u = scale (e^gc o U + sum_b e^(gc - ref_b) o (A Y)_b),   dp likewise with P0, B
//   p = e^(u - lse),   du = p (dp - delta) + dlse_gsa e^(u - lse_gsa),   xg += du u + p dp
//   X_b = scale du o e^(gc - ref_b),   Xp_b = p o e^(gc - ref_b)
//   ck = X Y^T, cv = Xp Y^T (i >= r),   ds_intra += e^(ref - gc) o (A^T X + B^T Xp)
//   N_k += q^T X_0, N_v += do^T Xp_0,   dk'_intra += ck^T q, dv'_intra += cv^T do,   dq = X_0 hk0 + ck k'
// (N is the inhomogeneous term of the state-gradient recurrence.)
//
// Waves 0-3 hold the k side (q, k', hk), waves 4-7 the v side (do, v', hv); a wave owns 16 columns (rows j, r or slots m) of
// every 64 x 64 table.  u and dp trade sides through LDS once per head; every table lies transposed ([column][row]), so
// that an accumulator's four rows are one 8-byte write and both operand forms are reads of it (plain or transposing).
//
// Bound, several query heads per kv-head: latency between short products -- one workgroup of eight waves fits a CU (LDS), a head
// is eight barriers with 4 to 100 MFMAs per wave between them, about 21k cycles of which vector instructions are 11k and MFMAs 6k
// per SIMD; a workgroup's first loads (20k cycles, all CUs at once and so at the rate of the memory) and its results come on top.
// One query head per kv-head (ONE): bytes (B=8, T=2048, 4/4 heads of 256: 580 MB in 159 us, half of them the fp32 results).
// Times: 415 us at B=2, T=8192, 32/8 heads of 128 (and 7 for the launch that looks for strongly decaying chunks), 159 + 7 at B=8,
// T=2048, 4/4 heads of 256, 88 + 5 at 5003 packed tokens, 16/16 heads of 64.
//
// Registers are the scarce thing: sums over the heads (64 at DW = 128) and the operands (48) stay, so whatever spills waits,
// with every load before it, for memory.  Hence: nothing derived from the lane's number lives across the loop over heads;
// wave-uniform bases with 32-bit offsets; Y read from LDS in both forms; stores only after the last load; the rows of o in whole
// lines, 8 of them to each wave, instead of in the layout of the products by half of the waves (456 -> 415 us at the first shape:
// 16 registers and the spills with them, and the half that had no rows waited), and N with its slots along the registers, so that a
// lane's four sums are one store.  Operands staged through LDS in whole lines, which other kernels gain from, change nothing here.
//
// Precision: dg is a difference of nearly equal sums, so every table made from fp32 values (X, Xp, Y, ck, cv, the chunk-start
// states) is a bf16 pair hi + lo and its products are hi hi + hi lo + lo hi (single bf16 tables put 1-5 % on dg).
#include "mfma_common.h"

namespace nha {
namespace {

using namespace mf;

// keeps the scheduler from collecting the operand reads of a whole unrolled stage in registers
#define FENCE __builtin_amdgcn_sched_barrier(0)

// Row strides (bf16).  The tables are read and written 8 bytes per lane, along rows and transposed; the tiles are read 16
// bytes per lane of 16 rows and transposed.  LDS cycles of a wave instruction with eight waves at it: tile rows 8.1 at D + 8,
// 4.15 at D + 16; tiles transposed 4.4 / 3.3; tables written transposed 8.1 at 72, 6.4 at 68, read so 3.3 / 4.5, transposing
// read 4.4 / 4.5.  68 is what leaves room for the tiles' D + 16.
constexpr int TLD = 68;    // 64 x 64 tables
constexpr int HLD = 36;    // tables that hold rows 32..63 only

__device__ __forceinline__ float logaddexp_f(float a, float b) {
  const float mx = fmaxf(a, b);
  return mx + logf(expf(a - mx) + expf(b - mx));
}

// 8 rows of column n of a transposed table tab[n][row]: rows r0 + 4 kb + e and r0 + 16 + 4 kb + e (the numbering of a
// transposing read of [row][n], lds_frag_tr)
__device__ __forceinline__ bf16x8 col_frag(const lbf16* tab, int ld, int n, int r0, int kb) {
  struct { bf16x4 a, b; } t;
  t.a = *reinterpret_cast<const NHA_LDS bf16x4*>(tab + n * ld + r0 + 4 * kb);
  t.b = *reinterpret_cast<const NHA_LDS bf16x4*>(tab + n * ld + r0 + 16 + 4 * kb);
  return __builtin_bit_cast(bf16x8, t);
}
__device__ __forceinline__ void put4(lbf16* p, const f32x4& v) {
  bf16x4 h;
#pragma unroll
  for (int e = 0; e < 4; ++e) h[e] = (__bf16)v[e];
  *reinterpret_cast<NHA_LDS bf16x4*>(p) = h;
}
// x as a bf16 pair
__device__ __forceinline__ void put4_pair(lbf16* hi, lbf16* lo, int idx, const f32x4& v) {
  bf16x4 h, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    h[e] = (__bf16)v[e];
    l[e] = (__bf16)(v[e] - (float)h[e]);
  }
  *reinterpret_cast<NHA_LDS bf16x4*>(hi + idx) = h;
  *reinterpret_cast<NHA_LDS bf16x4*>(lo + idx) = l;
}

// x of another lane of the row of 16
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

// element at a 32-bit byte offset of a base that is the same for the whole wave (one scalar and one vector register)
template <class T, class B>
__device__ __forceinline__ T ld_at(const B* base, unsigned bytes) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + bytes);
}
template <class T, class B>
__device__ __forceinline__ void st_at(B* base, unsigned bytes, const T& v) {
  *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + bytes) = v;
}

struct SlotP {
  const bf16_t *q, *dout, *o, *kg, *v, *s;     // q_gsa, dout, o [T,HQ,D]; k_gsa, v [T,H,D]; s [T,H,64]
  const float *lse_swa, *lse_gsa, *dlse_gsa;   // [T,HQ]
  const bf16_t *hk, *hv;                       // [NT][H][64][D] segment-local chunk-start states
  const float *hsk, *hsv;                      // [segment slot][H][64][D] segment-start states
  const float *dcum, *gc;                      // [NT][H][64] decay since the segment start, [NT][H][64][64] gate cumsums
  const int32_t *cu, *cidx, *coff;
  bf16_t* dq;                                  // dq_gsa [T,HQ,D]
  float *delta;                                // [T,HQ]
  float *xg, *dsi;                             // [T,H,64] (row token)
  float *ek, *ev;                              // [NT][H][D][64]
  float *dks, *dvs;                            // [T,H,D] (source token)
  int64_t pm, pe, pd;                          // floats between the sums of two parts of a kv-head's query heads: xg, dsi; ek, ev; dks, dvs
  int HQ, H, NG, NT, shift, seg_sh;            // NG: query heads of a workgroup (a kv-head's are shared out over gridDim.z)
  float scale;
};

template <int DW, bool ONE> struct SlotLds {
  static constexpr int LDT = DW + 16, TILE = BT * LDT, TAB = BT * TLD, HTAB = BT * HLD;
  static constexpr int Q = 0, O = Q + TILE;     // bf16 offsets
  static constexpr int X0 = O + TILE;           // X0 hi, lo, Xp0 hi, lo   [64 m][TLD]; u / dp in transit
  static constexpr int A = X0 + 4 * TAB;        // A, B [64 j][TLD], then X1 hi, lo, Xp1 hi, lo [64 m][HLD]
  static constexpr int X1 = A + 2 * TAB;
  static constexpr int C = A;                   // ck hi, lo, cv hi, lo [64 r][TLD], once A, B, X1, Xp1 are done with
  // k-state [64 m][LDT], k' [64 j][LDT]; first the other columns of q and do (ONE: where q and do were, once N and out are formed)
  static constexpr int S = ONE ? Q : X1 + 4 * HTAB;
  static constexpr int ROW = X1 + 4 * HTAB + (ONE ? 0 : 2 * TILE);   // floats: delta, lse, lse_gsa, dlse_gsa of the 64 rows
  static constexpr int Y = ROW + 2 * 4 * BT;                    // Y hi, lo [64 j][TLD]
  static constexpr size_t BYTES = (size_t)(Y + 2 * TAB) * 2;
  static_assert(2 * TAB <= 4 * HTAB, "ck and cv fit where A, B, X1 and Xp1 were");
  static_assert(BYTES <= 160 * 1024, "LDS");
};

// A contraction step's operands of one side for row / slot col: k' or v' and the chunk-start state (local + segment part);
// the loads, then the forms the products take (the state as a bf16 pair).
struct Operands {
  uint4 a, b;
  float4 c, d;
  __device__ __forceinline__ void load(const bf16_t* y, unsigned ybytes, const bf16_t* h, const float* s, unsigned index, int x) {
    a = ld_at<uint4>(y + x, ybytes);
    b = ld_at<uint4>(h + x, 2 * index);
    c = ld_at<float4>(s + x, 4 * index);
    d = ld_at<float4>(s + x + 4, 4 * index);
  }
  __device__ __forceinline__ void form(bool live, float dec, bf16x8& y, bf16x8& hi, bf16x8& lo) const {
    y = as_bf16x8(live ? a : make_uint4(0, 0, 0, 0));
    const bf16x8 l = as_bf16x8(b);
    const float s[8] = {c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = (float)l[e] + s[e] * dec;
      hi[e] = (__bf16)x;
      lo[e] = (__bf16)(x - (float)hi[e]);
    }
  }
};

// EXACT: the chunks in which some slot decays by more than e^-BWD_DECAY_CLAMP within a 32-row half (the growing factor of the
// split decay would leave the range); the other launch skips them.  Pairs of rows in different 16-row blocks take the cumsum
// at the start of the later row's block as their reference, both factors then shrink (Tb: X and Xp against their own block);
// pairs within a block have their decay formed one by one in fp32.  With all pairs of the chunk one by one this launch was slower
// than the VALU kernels that it replaced: backward of 4000 tokens, every chunk strongly decaying, 32/8 heads of 128 1985 us with
// those, 2702 with all pairs, 1142 like this; 3000 tokens, 4 heads of 256 525 / 802 / 413; 5000, 16 of 64 1040 / 1735 / 720.
// ONE: one query head per kv-head.  Nothing is summed over heads, so N and out leave the products as they are formed (no sums in
// registers), and the tiles of dq take the place of q and do once those are done with: a workgroup has all columns, also the 256
// of the largest head, and requests all of its operands at once (240 -> 159 us at B=8, T=2048, 4/4 heads of 256, where two
// workgroups of 128 columns each had formed the tables; 96 -> 88 at 5003 packed tokens, 16/16 heads of 64).
// DW: the output columns x of a workgroup.  With several heads half of the 256 of the largest head: a workgroup of all would hold
// 128 sums per lane next to its operands and tiles of 66 KB; the products over all columns (A, B, U, P0, delta) are formed twice
// instead, from the other columns of q and do in the room of the state tiles and operands streamed two steps at a time.
template <int D, int DW, bool EXACT, bool ONE>
__global__ __launch_bounds__(512) void bwd_slot_kernel(const SlotP p) {
  static_assert(!ONE || (D == DW && !EXACT), "ONE: all columns, split decays");
  typedef SlotLds<DW, ONE> L;
  constexpr int KS = D / 32, KW = DW / 32, DB = DW / 16, LDT = L::LDT;
  constexpr int NPC = BT * DW / 8 / 256;   // 16-byte pieces of a tile per thread of the side
  constexpr int LO = D / 8, NO = D / 64;   // lanes to a row of o, pieces of a lane of the wave's 8 rows
  constexpr bool KEEP = D == DW;   // the operands, the same for every head, stay in registers
  extern __shared__ __align__(16) unsigned char smem[];
  lbf16* const sm = (lbf16*)smem;
  const int tid = threadIdx.x, lane0 = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave & 3;
  const bool vs = wave >= 4;
  const int H = p.H, HQ = p.HQ, NG = p.NG, part = ONE ? 0 : blockIdx.z;
  // Several heads of 128 columns, two rounds of workgroups or more: the 32 CUs of an XCD start 0.2 us after one another (the second round
  // follows from the first).  All in step, their products come at the same moments, and two of the three cards that this was measured on
  // then run every matrix kernel of the following milliseconds up to 5 % slower, at the same clock: steps of 2 x 8192 tokens, 32 / 8 heads of 128, W =
  // 2048 one after another 2950 -> 2740 us, W = 512 1686 -> 1565, 5000 tokens 666 -> 640 (0.1 us 641, 2820 and 1615; 0.4 us 2735 and 1563).
  // On the second 2748 -> 2712, 1595 -> 1516, 630 -> 624; on the third 2658 -> 2657, 1512 -> 1506, 623 -> 622.  4 x 4096 tokens, 8 / 2
  // heads of 256: 957 on all.  Not at head size 64, where it only costs (2 x 4096 tokens, 16 / 4 heads, W = 300 282.4 -> 284.4), nor in one
  // round (2001 tokens 273 -> 280 us).
  if (D >= 128 && !ONE && !EXACT && gridDim.x * gridDim.y >= 512) {
    const unsigned L = blockIdx.y * gridDim.x + blockIdx.x;
    if (L < 256)
      for (unsigned i = 0; i < L >> 3; ++i) __builtin_amdgcn_s_sleep(8);
  }
  int h, chunk;
  xcd_tile(D / DW, p.NT, h, chunk);
  const int x0 = (h % (D / DW)) * DW;
  h /= D / DW;
  const int hq0 = ONE ? h : (h * gridDim.z + part) * NG;   // the workgroup's first query head
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1], c0 = bos + it * BT;
  const int R = (eos - c0) < BT ? (eos - c0) : BT;
  const int64_t cg = (int64_t)chunk * H + h;
  const int64_t sl = (int64_t)seg_slot(p.coff, n, it, p.seg_sh) * H + h;
  const float* const gc = p.gc + cg * BT * MS;   // rows past R repeat the last one
  int vlo = p.shift - it * BT;   // rows before vlo have no source token
  vlo = vlo < 0 ? 0 : vlo;
  const int tl0 = it * BT - p.shift > 0 ? it * BT - p.shift : 0;   // first source token a row may have

  lbf16* const X = sm + (vs ? L::O : L::Q);                      // this side's tile
  lbf16* const Z = sm + L::S + (vs ? L::TILE : 0);               // its other columns (until the state tiles are written)
  lbf16* const T0h = sm + L::X0 + (vs ? 2 * L::TAB : 0), * const T0l = T0h + L::TAB;   // X0 or Xp0
  lbf16* const T1h = sm + L::X1 + (vs ? 2 * L::HTAB : 0), * const T1l = T1h + L::HTAB;
  lbf16* const Tbh = sm + (vs ? L::Y : L::X1), * const Tbl = Tbh + L::TAB;   // EXACT has neither Y nor X1
  lbf16* const AT = sm + L::A + (vs ? L::TAB : 0);               // A or B
  lbf16* const Ch = sm + L::C + (vs ? 2 * L::TAB : 0), * const Cl = Ch + L::TAB;
  lfloat* const rdelta = (lfloat*)(NHA_LDS void*)(sm + L::ROW), * const rlse = rdelta + BT, * const rlg = rlse + BT, * const rdlg = rlg + BT;
  const lbf16* const Yh = sm + L::Y, * const Yl = Yh + L::TAB;
  lfloat* const transit = (lfloat*)(NHA_LDS void*)(sm + L::X0);   // [side][w][blk][lane] four floats

  // columns of a contraction step: the workgroup's own last
  auto step_col = [&](int ks) { return KEEP ? 32 * ks : ks < KW ? (x0 ^ DW) + 32 * ks : x0 + 32 * (ks - KW); };
  auto step_tile = [&](int ks) { return KEEP ? X + 32 * ks : ks < KW ? Z + 32 * ks : X + 32 * (ks - KW); };
  // ---- per head: the side's tile, the o rows of delta, the rows' log-sum-exps ---------------------------------------
  // (rows past R repeat the last one: their X and Xp are zero, whatever their scores)
  struct Head {
    uint4 x[NPC], z[KEEP ? 1 : NPC];
    float ls, lg, dl;
  };
  struct Rows {
    uint4 o[NO];
  };
  auto load_head = [&](Head& t, int hq, int lane) {
    const int stid = 64 * w + lane;
    const bf16_t* src = (vs ? p.dout : p.q) + ((int64_t)c0 * HQ + hq) * D;
#pragma unroll
    for (int u = 0; u < NPC; ++u) {
      const unsigned c = stid + 256 * u;
      const int row = c / (DW / 8), cc = (c % (DW / 8)) * 8;
      const unsigned at = ((row < R ? row : R - 1) * HQ * D + cc) * 2;
      t.x[u] = ld_at<uint4>(src + x0, at);
      if constexpr (!KEEP) t.z[u] = ld_at<uint4>(src + (x0 ^ DW), at);
    }
    if (!vs && w == 0) {
      const int64_t tq = (int64_t)(c0 + (lane < R ? lane : R - 1)) * HQ + hq;
      t.ls = p.lse_swa[tq];
      t.lg = p.lse_gsa[tq];
      t.dl = p.dlse_gsa ? p.dlse_gsa[tq] : 0.f;
    }
  };
  auto load_o = [&](Rows& t, int hq, int lane) {
    const bf16_t* const src = p.o + ((int64_t)c0 * HQ + hq) * D;
#pragma unroll
    for (int u = 0; u < NO; ++u) {
      const int row = 8 * wave + 8 / NO * u + lane / LO;
      t.o[u] = ld_at<uint4>(src, ((row < R ? row : R - 1) * HQ * D + 8 * (lane % LO)) * 2);
    }
  };
  auto row_delta = [&](const Rows& t, int hq, int lane) {
#pragma unroll
    for (int u = 0; u < NO; ++u) {
      const int row = 8 * wave + 8 / NO * u + lane / LO, c = 8 * (lane % LO);
      const lbf16* const dp = KEEP || (c & DW) == (x0 & DW) ? sm + L::O + row * LDT + c % DW : sm + L::S + L::TILE + row * LDT + c % DW;
      const bf16x8 o8 = as_bf16x8(t.o[u]), d8 = *reinterpret_cast<const NHA_LDS bf16x8*>(dp);
      float acc = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc += (float)o8[e] * (float)d8[e];
      acc += dpp_f<0xB1>(acc);    // lanes 1 and 2 apart, the other four of 8, of 16, of 32
      acc += dpp_f<0x4E>(acc);
      acc += dpp_f<0x141>(acc);
      if (LO >= 16) acc += dpp_f<0x140>(acc);
      if (LO >= 32) acc += __shfl_xor(acc, 16, 64);
      if (lane % LO == 0) {
        rdelta[row] = acc;
        if (row < R && x0 == 0) p.delta[(int64_t)(c0 + row) * HQ + hq] = acc;
      }
    }
  };
  auto store_head = [&](const Head& t, int lane) {
    const int stid = 64 * w + lane;
#pragma unroll
    for (int u = 0; u < NPC; ++u) {
      const unsigned c = stid + 256 * u;
      const int row = c / (DW / 8), cc = (c % (DW / 8)) * 8;
      lds_st16(X + row * LDT + cc, t.x[u]);
      if constexpr (!KEEP) lds_st16(Z + row * LDT + cc, t.z[u]);
    }
    if (wave == 0) {
      rlse[lane] = logaddexp_f(t.ls, t.lg);
      rlg[lane] = t.lg;
      rdlg[lane] = t.dl;
    }
  };
  Rows orow;
  float gi[4][4], g31;   // gate cumsums of a lane's rows 16 blk + 4 kb + e (slot col)
  auto load_gates = [&](int kb, int col) {
#pragma unroll
    for (int blk = 0; blk < 4; ++blk)
#pragma unroll
      for (int e = 0; e < 4; ++e) gi[blk][e] = ld_at<float>(gc + (16 * blk + e) * MS, (4 * kb * MS + col) * 4);
    g31 = ld_at<float>(gc + 31 * MS, col * 4);
  };
  float e0[4][4], e1[2][4];   // their exponentials, of the rows 32.. also against the cumsum at row 31
  Operands opd[KEEP ? KS : 2];
  auto load_operands = [&](int x, int ks, int lane) {
    const int l16 = lane & 15, kb = lane >> 4, col = 16 * w + l16;
    const int tl = it * BT + col - p.shift;
    const bool has = col < R && tl >= 0;
    const unsigned index = col * D + 8 * kb;
    opd[x].load((vs ? p.v : p.kg) + ((int64_t)(bos + tl0) * H + h) * D, ((has ? tl - tl0 : 0) * H * D + 8 * kb) * 2,
                (vs ? p.hv : p.hk) + cg * MS * D, (vs ? p.hsv : p.hsk) + sl * MS * D, index, step_col(ks));
  };

  // ---- everything the first head needs is requested at once; whether the chunk is this launch's is known later, but in
  // the rare launch, which leaves at once
  const float g31t = gc[31 * MS + lane0], g63t = gc[63 * MS + lane0];
  auto mine = [&] { return (__any(g31t < -BWD_DECAY_CLAMP || g63t - g31t < -BWD_DECAY_CLAMP) != 0) == EXACT; };
  if (EXACT && !mine()) return;
  bf16x8 y[KEEP ? KS : 1], hh[KEEP ? KS : 1], hl[KEEP ? KS : 1];
  auto store_states = [&](int x, const bf16x8& hi, const bf16x8& yy, int lane) {   // the tiles of dq, from the k side
    lbf16* const at = sm + L::S + (16 * w + (lane & 15)) * LDT + x + 8 * (lane >> 4);
    *reinterpret_cast<NHA_LDS bf16x8*>(at) = hi;
    *reinterpret_cast<NHA_LDS bf16x8*>(at + L::TILE) = yy;
  };
  {
    const int l16 = lane0 & 15, kb = lane0 >> 4, col = 16 * w + l16;
    const int j = tid >> 3, m8 = (tid & 7) * 8;
    const bool live = j >= vlo && j < R;
    float sv[8], g[8], ref[8];
    Elem<bf16_t>::ld8(p.s + (((int64_t)(live ? c0 + j - p.shift : bos)) * H + h) * MS + m8, sv);
    Elem<float>::ld8(gc + j * MS + m8, g);
    Elem<float>::ld8(gc + 31 * MS + m8, ref);
    Head head;
    load_head(head, hq0, lane0);
    if constexpr (ONE) load_o(orow, hq0, lane0);
    const float dc = p.dcum[cg * MS + col];
#pragma unroll
    for (int ks = 0; ks < (KEEP ? KS : 2); ++ks) load_operands(ks, ks, lane0);
    FENCE;
    if (!EXACT && !mine()) return;
    if constexpr (!EXACT)
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      f32x4 yv;
#pragma unroll
      for (int x = 0; x < 4; ++x) yv[x] = live ? sv[e + x] * __expf((j >= 32 ? ref[e + x] : 0.f) - g[e + x]) : 0.f;
      put4_pair(sm + L::Y, sm + L::Y + L::TAB, j * TLD + m8 + e, yv);
    }
    store_head(head, lane0);
    if constexpr (KEEP) {
      const int tl = it * BT + col - p.shift;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        opd[ks].form(col < R && tl >= 0, dc, y[ks], hh[ks], hl[ks]);
        if (!ONE && !vs) store_states(32 * ks, hh[ks], y[ks], lane0);
      }
    }
    if constexpr (ONE) {
      load_gates(kb, col);
#pragma unroll
      for (int blk = 0; blk < 4; ++blk)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          e0[blk][e] = __expf(gi[blk][e]);
          if (blk >= 2) e1[blk - 2][e] = __expf(gi[blk][e] - g31);
        }
    }
    lds_barrier();
  }
  f32x4 accN[ONE ? 1 : DB], accO[ONE ? 1 : DB], accS[4], xg[2];   // xg: of the rows 32.. on the v side, of the others on the k side
#pragma unroll
  for (int d = 0; d < (ONE ? 1 : DB); ++d) accN[d] = accO[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) accS[rb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  xg[0] = xg[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float* const ep = (vs ? p.ev : p.ek) + part * p.pe + (cg * D + x0) * MS;            // N [x][m]
  float* const op = (vs ? p.dvs : p.dks) + part * p.pd + ((int64_t)(bos + tl0) * H + h) * D + x0;   // out, at the rows' source tokens

  // xg and ds_intra (the sum of both sides): rows 32.. from the v side, the others from the k side
  lfloat* const sums = ONE ? (lfloat*)(NHA_LDS void*)(sm + L::Y) : transit;
  auto swap_sums = [&](int lane) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (vs) {   // (swapped in place: a choice between two elements by reference would put the array in memory)
        const f32x4 z = accS[b];
        accS[b] = accS[2 + b];
        accS[2 + b] = z;
      }
      *reinterpret_cast<NHA_LDS f32x4*>(sums + ((wave * 2 + b) * 64 + lane) * 4) = accS[2 + b];
    }
  };
  auto store_sums = [&](int kb, int col, int lane) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const f32x4 z = accS[b] + *reinterpret_cast<const NHA_LDS f32x4*>(sums + (((wave ^ 4) * 2 + b) * 64 + lane) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 16 * b + 4 * kb + e + (vs ? 32 : 0);
        const unsigned at = (r * H * MS + col) * 4;
        const float d = vs ? g31 - gi[2 + b][e] : -gi[b][e];
        if (r < R) {
          st_at(p.xg + part * p.pm + ((int64_t)c0 * H + h) * MS, at, xg[b][e]);
          st_at(p.dsi + part * p.pm + ((int64_t)c0 * H + h) * MS, at, EXACT ? z[e] : z[e] * __expf(d));
        }
      }
    }
  };
  auto store_sides = [&](int d, const f32x4& n, const f32x4& o, int lane) {
    const int l16 = lane & 15, kb = lane >> 4, col = 16 * w + l16, tl = it * BT + col - p.shift;
    st_at(ep + 16 * d * MS + 16 * w, (l16 * MS + 4 * kb) * 4, n);
    if (col < R && tl >= 0) st_at(op + 16 * d, ((tl - tl0) * H * D + 4 * kb) * 4, o);
  };
  for (int a = 0; a < (ONE ? 1 : NG); ++a) {
    const int hq = hq0 + a;
    // what depends on the lane's number is derived anew for every head: hoisted out of the loop, the addresses and decay
    // factors of a whole head are kept across it -- in memory, there are no registers for them
    int lane = lane0;
    asm volatile("" : "+v"(lane));
    const int l16 = lane & 15, kb = lane >> 4, col = 16 * w + l16;
    if constexpr (!ONE) load_o(orow, hq, lane);
    if constexpr (!KEEP) row_delta(orow, hq, lane);
    FENCE;
    // ---- A or B (rows 16 blk + 4 kb + e, column j = col), U or P0 (slot m = col) --------------------------------------
    f32x4 cU[4];
    auto put_scores = [&](int blk, f32x4 c) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (16 * blk + 4 * kb + e < col) c[e] = 0.f;   // j <= i
      put4(AT + col * TLD + 16 * blk + 4 * kb, c);
    };
    if constexpr (ONE) {
      f32x4 cA[4];
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) cA[blk] = cU[blk] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) {
          const bf16x8 x = lds_frag(X, LDT, 16 * blk + l16, 32 * ks + 8 * kb);
          cA[blk] = mfma16(x, y[ks], cA[blk]);
          cU[blk] = mfma16(x, hh[ks], mfma16(x, hl[ks], cU[blk]));
        }
        if (ks % 2 == 1) FENCE;
      }
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) put_scores(blk, cA[blk]);
    } else if constexpr (KEEP) {
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) {
        f32x4 cA = {0.f, 0.f, 0.f, 0.f};
        cU[blk] = cA;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const bf16x8 x = lds_frag(X, LDT, 16 * blk + l16, 32 * ks + 8 * kb);
          cA = mfma16(x, y[ks], cA);
          cU[blk] = mfma16(x, hh[ks], mfma16(x, hl[ks], cU[blk]));
        }
        put_scores(blk, cA);
        FENCE;
      }
    } else {
      f32x4 cA[4];
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) cA[blk] = cU[blk] = (f32x4){0.f, 0.f, 0.f, 0.f};
      const float dc = p.dcum[cg * MS + col];
      const int tl = it * BT + col - p.shift;
      const bool has = col < R && tl >= 0;
      // a pair of steps is requested while the pair before it is in the products
#pragma unroll
      for (int ks = 0; ks < KS; ks += 2) {
        bf16x8 yy[2], hi[2], lo[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          opd[x].form(has, dc, yy[x], hi[x], lo[x]);
          if (ks >= KW && !vs) store_states(32 * (ks - KW + x), hi[x], yy[x], lane);
        }
        FENCE;
        if (ks + 2 < KS)
#pragma unroll
          for (int x = 0; x < 2; ++x) load_operands(x, ks + 2 + x, lane);
        FENCE;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int blk = 0; blk < 4; ++blk) {
            const bf16x8 q8 = lds_frag(step_tile(ks + x), LDT, 16 * blk + l16, 8 * kb);
            cA[blk] = mfma16(q8, yy[x], cA[blk]);
            cU[blk] = mfma16(q8, hi[x], mfma16(q8, lo[x], cU[blk]));
          }
          FENCE;
        }
        if (ks + 2 == KW) lds_barrier();   // the other columns of q and do are done with
      }
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) put_scores(blk, cA[blk]);
    }
    if constexpr (!ONE) load_gates(kb, col);
    lds_barrier();
    // ---- u (k side) or dp (v side) of rows 16 blk + 4 kb + e, slot col, to the other side ------------------------------
    if constexpr (!EXACT) {
      bf16x8 yf[2][2];
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        yf[hf][0] = lds_frag_tr(Yh, TLD, 32 * hf, 32 * hf + 16, 16 * w, lane);
        yf[hf][1] = lds_frag_tr(Yl, TLD, 32 * hf, 32 * hf + 16, 16 * w, lane);
      }
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) {
        f32x4 c[2];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          c[hf] = (f32x4){0.f, 0.f, 0.f, 0.f};
          if (2 * hf > blk) continue;   // rows of the first half see none of the second
          const bf16x8 x = lds_frag_tr(AT, TLD, 32 * hf, 32 * hf + 16, 16 * blk, lane);
          c[hf] = mfma16(x, yf[hf][0], mfma16(x, yf[hf][1], c[hf]));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (!ONE) {
            e0[blk][e] = __expf(gi[blk][e]);
            if (blk >= 2) e1[blk - 2][e] = __expf(gi[blk][e] - g31);
          }
          cU[blk][e] = e0[blk][e] * (cU[blk][e] + c[0][e]) + (blk >= 2 ? e1[blk - 2][e] * c[1][e] : 0.f);
        }
        FENCE;
      }
    } else {
      float sj[4][4];   // strengths of the rows 16 blk + 4 kb + e
#pragma unroll
      for (int blk = 0; blk < 4; ++blk)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = 16 * blk + 4 * kb + e;
          const bool on = j >= vlo && j < R;
          const float x = bf16_to_f32(p.s[((int64_t)(on ? c0 + j - p.shift : bos) * H + h) * MS + col]);
          sj[blk][e] = on ? x : 0.f;
        }
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) {
        f32x4 c = {0.f, 0.f, 0.f, 0.f};
        const float ref = blk ? ld_at<float>(gc + (16 * blk - 1) * MS, col * 4) : 0.f;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {   // earlier blocks against ref
          if (2 * hf >= blk) continue;
          bf16x8 yh, yl;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int bj = 2 * hf + (e >> 2);
            const float y = bj < blk ? sj[bj][e & 3] * expf(ref - gi[bj][e & 3]) : 0.f;
            yh[e] = (__bf16)y;
            yl[e] = (__bf16)(y - (float)yh[e]);
          }
          const bf16x8 x = lds_frag_tr(AT, TLD, 32 * hf, 32 * hf + 16, 16 * blk, lane);
          c = mfma16(x, yh, mfma16(x, yl, c));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) cU[blk][e] = expf(gi[blk][e]) * cU[blk][e] + (blk ? expf(gi[blk][e] - ref) * c[e] : 0.f);
#pragma unroll 4
        for (int jj = 0; jj < 16; ++jj) {   // the block itself (A is zero for rows before j, whose factor may leave the range)
          const int j = 16 * blk + jj;
          const bool on = j >= vlo && j < R;
          const float s = bf16_to_f32(p.s[((int64_t)(on ? c0 + j - p.shift : bos) * H + h) * MS + col]), gj = gc[j * MS + col];
          const bf16x4 a = *reinterpret_cast<const NHA_LDS bf16x4*>(AT + j * TLD + 16 * blk + 4 * kb);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = (float)a[e] * s * expf(gi[blk][e] - gj);
            cU[blk][e] += on && 4 * kb + e >= jj ? x : 0.f;
          }
        }
        FENCE;
      }
    }
    if constexpr (KEEP) row_delta(orow, hq, lane);
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      if (!vs) cU[blk] *= p.scale;
      *reinterpret_cast<NHA_LDS f32x4*>(transit + ((wave * 4 + blk) * 64 + lane) * 4) = cU[blk];
    }
    lds_barrier();
    f32x4 other[4];
#pragma unroll
    for (int blk = 0; blk < 4; ++blk)
      other[blk] = *reinterpret_cast<const NHA_LDS f32x4*>(transit + (((wave ^ 4) * 4 + blk) * 64 + lane) * 4);
    lds_barrier();
    // ---- p, du; X or Xp into the tables, xg ---------------------------------------------------------------------------
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      const int i0 = 16 * blk + 4 * kb;
      const f32x4 lt = *reinterpret_cast<const NHA_LDS f32x4*>(rlse + i0), dl = *reinterpret_cast<const NHA_LDS f32x4*>(rdelta + i0);
      f32x4 u = vs ? other[blk] : cU[blk], dp = vs ? cU[blk] : other[blk], pm, du;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pm[e] = EXACT ? expf(u[e] - lt[e]) : __expf(u[e] - lt[e]);
        du[e] = pm[e] * (dp[e] - dl[e]);
      }
      if (p.dlse_gsa) {
        const f32x4 lg = *reinterpret_cast<const NHA_LDS f32x4*>(rlg + i0), dg = *reinterpret_cast<const NHA_LDS f32x4*>(rdlg + i0);
#pragma unroll
        for (int e = 0; e < 4; ++e) du[e] += dg[e] * (EXACT ? expf(u[e] - lg[e]) : __expf(u[e] - lg[e]));
      }
      f32x4 t0, t1;
      float own[4];
      if constexpr (EXACT)
#pragma unroll
        for (int e = 0; e < 4; ++e) own[e] = blk ? gi[blk][e] - ld_at<float>(gc + (16 * blk - 1) * MS, col * 4) : gi[blk][e];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = i0 + e < R ? (vs ? pm[e] : p.scale * du[e]) : 0.f;
        t0[e] = x * (EXACT ? expf(gi[blk][e]) : e0[blk][e]);
        if constexpr (EXACT) t1[e] = x * expf(own[e]);
        else if (blk >= 2) t1[e] = x * e1[blk - 2][e];
        if constexpr (EXACT) ep[(i0 + e) * MS + col] = x;   // undecayed, for the pairwise sums (N takes the place afterwards)
      }
      put4_pair(T0h, T0l, col * TLD + i0, t0);
      if constexpr (EXACT) put4_pair(Tbh, Tbl, col * TLD + i0, t1);
      else if (blk >= 2) put4_pair(T1h, T1l, col * HLD + i0 - 32, t1);
      if (vs == (blk >= 2)) xg[blk & 1] += du * u + pm * dp;
      FENCE;
    }
    if constexpr (EXACT) __syncthreads();   // (global stores of the side included)
    else lds_barrier();
    // ---- ck or cv: rows 16 blk + 4 kb + e, column r = col; ds_intra -----------------------------------------------------
    f32x4 c[4];
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) c[blk] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if constexpr (!EXACT) {
      // columns r of the first half take the tables with ref 0, the others those with gc_31 (rows >= 32 only: set back)
      const lbf16* const Tch = w < 2 ? T0h : T1h - 32, * const Tcl = w < 2 ? T0l : T1l - 32;
      const int tcld = w < 2 ? TLD : HLD;
      bf16x8 yf[2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        yf[ks][0] = col_frag(Yh, TLD, col, 32 * ks, kb);
        yf[ks][1] = col_frag(Yl, TLD, col, 32 * ks, kb);
      }
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) {
        if (blk < w) continue;   // i >= r
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const bf16x8 xh = lds_frag_tr(Tch, tcld, 32 * ks, 32 * ks + 16, 16 * blk, lane);
          const bf16x8 xl = lds_frag_tr(Tcl, tcld, 32 * ks, 32 * ks + 16, 16 * blk, lane);
          c[blk] = mfma16(xh, yf[ks][0], mfma16(xh, yf[ks][1], mfma16(xl, yf[ks][0], c[blk])));
        }
        FENCE;
      }
      // ds[r][m = col] += sum_i A[i][r] X[i][m]  (B, Xp on the v side): rows r of the first half against ref 0, the others
      // against gc_31 (they meet rows of the second half only)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const bf16x8 xh = col_frag(T0h, TLD, col, 32 * hf, kb), xl = col_frag(T0l, TLD, col, 32 * hf, kb);
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          const bf16x8 af = col_frag(AT, TLD, 16 * rb + l16, 32 * hf, kb);
          accS[rb] = mfma16(af, xh, mfma16(af, xl, accS[rb]));
        }
        FENCE;
      }
      const bf16x8 xh = col_frag(T1h, HLD, col, 0, kb), xl = col_frag(T1l, HLD, col, 0, kb);
#pragma unroll
      for (int rb = 2; rb < 4; ++rb) {
        const bf16x8 af = col_frag(AT, TLD, 16 * rb + l16, 32, kb);
        accS[rb] = mfma16(af, xh, mfma16(af, xl, accS[rb]));
      }
    } else {
      const int tl = it * BT + col - p.shift;
      const bool on = col < R && tl >= 0;
      const bf16_t* const sr = p.s + ((int64_t)(on ? bos + tl : bos) * H + h) * MS;
      // rows i of later blocks than r's: against the start of their block
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        float y[8], g[8];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int m = 32 * ks + 16 * q + 4 * kb;
          const bf16x4 sv = *reinterpret_cast<const bf16x4*>(sr + m);
          const f32x4 gv = *reinterpret_cast<const f32x4*>(gc + col * MS + m);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[4 * q + e] = on ? (float)sv[e] : 0.f, g[4 * q + e] = gv[e];
        }
#pragma unroll
        for (int blk = 1; blk < 4; ++blk) {
          if (blk <= w) continue;
          const f32x4 ra = *reinterpret_cast<const f32x4*>(gc + (16 * blk - 1) * MS + 32 * ks + 4 * kb);
          const f32x4 rb = *reinterpret_cast<const f32x4*>(gc + (16 * blk - 1) * MS + 32 * ks + 16 + 4 * kb);
          bf16x8 yh, yl;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float v = y[e] * expf((e < 4 ? ra[e & 3] : rb[e & 3]) - g[e]);
            yh[e] = (__bf16)v;
            yl[e] = (__bf16)(v - (float)yh[e]);
          }
          const bf16x8 xh = lds_frag_tr(Tbh, TLD, 32 * ks, 32 * ks + 16, 16 * blk, lane);
          const bf16x8 xl = lds_frag_tr(Tbl, TLD, 32 * ks, 32 * ks + 16, 16 * blk, lane);
          c[blk] = mfma16(xh, yh, mfma16(xh, yl, mfma16(xl, yh, c[blk])));
        }
        FENCE;
      }
      // rows i of r's block, four slots at a time
      f32x4 own = {0.f, 0.f, 0.f, 0.f};
      for (int m = 0; m < MS; m += 4) {
        const bf16x4 sv = *reinterpret_cast<const bf16x4*>(sr + m);
        const f32x4 gr = *reinterpret_cast<const f32x4*>(gc + col * MS + m);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 16 * w + 4 * kb + e;
          const f32x4 x = *reinterpret_cast<const f32x4*>(ep + i * MS + m), g = *reinterpret_cast<const f32x4*>(gc + i * MS + m);
          float z = 0.f;
#pragma unroll
          for (int u = 0; u < 4; ++u) z += x[u] * (float)sv[u] * expf(g[u] - gr[u]);
          own[e] += on && i >= col ? z : 0.f;
        }
      }
#pragma unroll
      for (int blk = 0; blk < 4; ++blk)
        if (blk == w) c[blk] = own;
      // ds_intra of rows r = 16 rb + 4 kb + e
#pragma unroll
      for (int bi = 1; bi < 4; ++bi) {
        bf16x8 xh = col_frag(Tbh, TLD, col, 32 * (bi >> 1), kb), xl = col_frag(Tbl, TLD, col, 32 * (bi >> 1), kb);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if ((e >> 2) != (bi & 1)) xh[e] = xl[e] = (__bf16)0.f;   // the other block of the half
        const float ref = ld_at<float>(gc + (16 * bi - 1) * MS, col * 4);
#pragma unroll
        for (int rb = 0; rb < bi; ++rb) {
          const bf16x8 af = col_frag(AT, TLD, 16 * rb + l16, 32 * (bi >> 1), kb);
          const f32x4 z = mfma16(af, xh, mfma16(af, xl, (f32x4){0.f, 0.f, 0.f, 0.f}));
#pragma unroll
          for (int e = 0; e < 4; ++e) accS[rb][e] += z[e] * expf(ref - gi[rb][e]);
        }
        FENCE;
      }
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) {
#pragma unroll 4
        for (int ii = 0; ii < 16; ++ii) {
          const int i = 16 * rb + ii;
          const float x = ep[i * MS + col], g = gc[i * MS + col];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float z = bf16_to_f32(AT[(16 * rb + 4 * kb + e) * TLD + i]) * x * expf(g - gi[rb][e]);
            accS[rb][e] += ii >= 4 * kb + e ? z : 0.f;
          }
        }
        FENCE;
      }
    }
    if constexpr (EXACT) __syncthreads();
    else lds_barrier();   // A, B, X1, Xp1 are done with
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (16 * blk + 4 * kb + e < col) c[blk][e] = 0.f;
      put4_pair(Ch, Cl, col * TLD + 16 * blk + 4 * kb, c[blk]);
    }
    if constexpr (ONE) swap_sums(lane);
    lds_barrier();
    if constexpr (ONE) store_sums(kb, col, lane);
    Head next = {};   // (a value on every path: left open, the registers count as live around the whole loop)
    if (!ONE && KEEP && a + 1 < NG) load_head(next, hq + 1, lane);
    FENCE;
    // ---- N (rows m = 16 w + 4 kb + e, columns x = 16 d + l16) and out^T: the tables times X ------------------------------
    if constexpr (ONE) {
      bf16x8 bw[2], bwl[2], bc[2], bcl[2];
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        bw[hf] = col_frag(T0h, TLD, col, 32 * hf, kb), bwl[hf] = col_frag(T0l, TLD, col, 32 * hf, kb);
        bc[hf] = col_frag(Ch, TLD, col, 32 * hf, kb), bcl[hf] = col_frag(Cl, TLD, col, 32 * hf, kb);
      }
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        f32x4 n = {0.f, 0.f, 0.f, 0.f}, o = n;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          const bf16x8 x = lds_frag_tr(X, LDT, 32 * hf, 32 * hf + 16, 16 * d, lane);
          n = mfma16(bw[hf], x, mfma16(bwl[hf], x, n));
          o = mfma16(x, bc[hf], mfma16(x, bcl[hf], o));
        }
        store_sides(d, n, o, lane);
        if (d % 2 == 1) FENCE;
      }
      lds_barrier();   // q and do are done with
      if (!vs)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) store_states(32 * ks, hh[ks], y[ks], lane);
      lds_barrier();
    } else {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const bf16x8 bw = col_frag(T0h, TLD, col, 32 * hf, kb), bwl = col_frag(T0l, TLD, col, 32 * hf, kb);
        const bf16x8 bc = col_frag(Ch, TLD, col, 32 * hf, kb), bcl = col_frag(Cl, TLD, col, 32 * hf, kb);
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          const bf16x8 x = lds_frag_tr(X, LDT, 32 * hf, 32 * hf + 16, 16 * d, lane);
          accN[d] = mfma16(bw, x, mfma16(bwl, x, accN[d]));
          accO[d] = mfma16(x, bc, mfma16(x, bcl, accO[d]));
          if (d % 2 == 1) FENCE;
        }
      }
    }
    FENCE;
    // ---- dq^T: rows i = 16 w + l16, this side's half of the columns -----------------------------------------------------
    {
      const lbf16* const Ht = sm + L::S, * const Kt = Ht + L::TILE;
      const lbf16* const W0h = sm + L::X0, * const W0l = W0h + L::TAB, * const Kh = sm + L::C, * const Kl = Kh + L::TAB;
      f32x4 acc[DB / 2];
#pragma unroll
      for (int d = 0; d < DB / 2; ++d) acc[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const bf16x8 bw = lds_frag_tr(W0h, TLD, 32 * hf, 32 * hf + 16, 16 * w, lane), bwl = lds_frag_tr(W0l, TLD, 32 * hf, 32 * hf + 16, 16 * w, lane);
        const bf16x8 bc = lds_frag_tr(Kh, TLD, 32 * hf, 32 * hf + 16, 16 * w, lane), bcl = lds_frag_tr(Kl, TLD, 32 * hf, 32 * hf + 16, 16 * w, lane);
#pragma unroll
        for (int d = 0; d < DB / 2; ++d) {
          const int c16 = 16 * d + (vs ? DW / 2 : 0);
          const bf16x8 x = lds_frag_tr(Ht, LDT, 32 * hf, 32 * hf + 16, c16, lane), k = lds_frag_tr(Kt, LDT, 32 * hf, 32 * hf + 16, c16, lane);
          acc[d] = mfma16(x, bw, mfma16(x, bwl, acc[d]));
          acc[d] = mfma16(k, bc, mfma16(k, bcl, acc[d]));
          if (d % 2 == 1) FENCE;
        }
      }
      if (col < R) {
        bf16_t* const dst = p.dq + ((int64_t)c0 * HQ + hq) * D + x0 + (vs ? DW / 2 : 0);
#pragma unroll
        for (int d = 0; d < DB / 2; ++d) {
          bf16x4 pk;
#pragma unroll
          for (int e = 0; e < 4; ++e) pk[e] = (__bf16)acc[d][e];
          st_at(dst + 16 * d, (col * HQ * D + 4 * kb) * 2, pk);
        }
      }
    }
    if (!ONE && a + 1 < NG) {
      if constexpr (!KEEP) load_head(next, hq + 1, lane);
      lds_barrier();   // the tiles and tables are done with
      store_head(next, lane);
      if constexpr (!KEEP) {
#pragma unroll
        for (int x = 0; x < 2; ++x) load_operands(x, x, lane);
      }
      lds_barrier();
    }
  }
  // ---- results (loads first: a load waits for the stores issued before it) ---------------------------------------------
  if constexpr (!ONE) {
    const int l16 = lane0 & 15, kb = lane0 >> 4, col = 16 * w + l16;
    if (x0 == 0) {
      load_gates(kb, col);
      lds_barrier();
      swap_sums(lane0);
      lds_barrier();
      store_sums(kb, col, lane0);
    }
#pragma unroll
    for (int d = 0; d < DB; ++d) store_sides(d, accN[d], accO[d], lane0);
  }
}

template <int D, int DW, bool EXACT, bool ONE>
int launch_one(const SlotP& p, hipStream_t st) {
  constexpr size_t lds = SlotLds<DW, ONE>::BYTES;
  static std::atomic<bool> configured{false};   // the attribute call is idempotent: a second thread may repeat it
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute((const void*)bwd_slot_kernel<D, DW, EXACT, ONE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      set_error("nha_prefill_bwd: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
      return NHA_ERR_LAUNCH;
    }
    configured = true;
  }
  hipLaunchKernelGGL((bwd_slot_kernel<D, DW, EXACT, ONE>), dim3(p.H * (D / DW), p.NT, p.HQ / (p.H * p.NG)), dim3(512), lds, st, p);
  NHA_CHECK_LAUNCH("nha_prefill_bwd(slot branch)");
  return NHA_OK;
}
template <int D>
int launch(const SlotP& p, hipStream_t st) {
  constexpr int DW = D < 128 ? D : 128;
  const int rc = p.HQ == p.H ? launch_one<D, D, false, true>(p, st) : launch_one<D, DW, false, false>(p, st);
  return rc != NHA_OK ? rc : launch_one<D, DW, true, false>(p, st);
}

}  // namespace

// A workgroup walks its query heads one after the other, 8 to 9 us each, so where the chunks and kv-heads of a call leave CUs without
// work the heads are shared out, as many ways as all workgroups still have a place at once; the scan over the chunks adds up the parts'
// sums.  32 / 4 heads of 128, us: 2 x 533 tokens (72 groups) 80 -> 49, the scan 5.3 -> 9.5; 2000 (128) 87 -> 53; forward and backward of
// the first at W = 950 308 -> 281.  With two rounds of smaller workgroups a call would pay their first loads (14 us) twice.
int bwd_slot_parts(const NhaPrefillBwdArgs* a) {
  const int NG = a->HQ / a->H;
  const int64_t groups = (int64_t)a->H * a->NT * (a->K == 256 ? 2 : 1);
  int parts = 1;
  while (parts < 8 && NG % (2 * parts) == 0 && 2 * parts * groups <= 256) parts *= 2;
  return parts;
}

int bwd_slot_branch(const NhaPrefillBwdArgs* a, const mf::MP& m, float* delta, float* xg, float* dsi, float* ek, float* ev, float* dks,
                    float* dvs, int parts) {
  SlotP p;
  p.q = (const bf16_t*)a->q_gsa; p.dout = (const bf16_t*)a->dout; p.o = (const bf16_t*)a->o;
  p.kg = (const bf16_t*)a->k_gsa; p.v = (const bf16_t*)a->v; p.s = (const bf16_t*)a->s;
  p.lse_swa = a->lse_swa; p.lse_gsa = a->lse_gsa; p.dlse_gsa = a->dlse_gsa;
  p.hk = m.hkT; p.hv = m.hvc; p.hsk = m.hseg_k; p.hsv = m.hseg_v; p.dcum = m.dcum; p.gc = m.gc;
  p.cu = a->cu_seqlens; p.cidx = a->chunk_indices; p.coff = a->chunk_offsets;
  p.dq = (bf16_t*)a->dq_gsa; p.delta = delta; p.xg = xg; p.dsi = dsi; p.ek = ek; p.ev = ev; p.dks = dks; p.dvs = dvs;
  p.HQ = a->HQ; p.H = a->H; p.NG = a->HQ / a->H / parts; p.NT = a->NT; p.shift = a->shift; p.seg_sh = m.seg_sh; p.scale = a->scale;
  p.pm = (int64_t)a->T_tot * a->H * MS; p.pe = (int64_t)a->NT * a->H * a->K * MS; p.pd = (int64_t)a->T_tot * a->H * a->K;
  hipStream_t st = (hipStream_t)a->stream;
  if (a->K == 64) return launch<64>(p, st);
  if (a->K == 128) return launch<128>(p, st);
  return launch<256>(p, st);
}

}  // namespace nha
