// fp32 NHA prefill on the fp32 matrix cores of gfx950 (v_mfma_f32_16x16x4_f32): K == V == D in {64,128,256}, M == 64, any
// grouping, window, shift, varlen.  Same op as prefill_simple.hip (which keeps every other shape) with no precision given
// up: fp32 operands, products and sums, exact decays.
//
//   state_local : per (chunk, kv-head, state) the chunk's own contribution  U = K^T (S exp(gc_last - gc)), [m][d], and the
//                 chunk-local gate cumsum gc
//   state_scan  : h_c+1 = exp(gc_last) h_c + U_c element by element over the chunks of a sequence; U_c is replaced by h_c
//   out         : one WAVE per (16 rows of a chunk, query head): window, slot logits, slot read, one softmax; four waves where
//                 there are few such units
//
// The generic kernels walk a sequence's chunks in one workgroup per 16 slots, every row's loads waited for one by one
// (115 us per chunk), and their output pass redoes the slot algebra per token; here the chunks are independent but for
// an element-wise scan, and everything else is matrix products.  Bound: launches and latencies at prompt sizes (B=1, T=512, 4
// heads of 64, W=64: 1028 -> 23 us of kernels), the fp32 matrix rate beyond (per call, generic kernels / these: B=1, T=2048,
// 8/2 heads of 128, W=64 8.2 ms / 62 us; B=2, T=4096, 32/8 heads 30.7 / 0.57 ms = 46 TFLOP/s; B=1, T=4096, 16 heads of 64,
// W=1024 16.9 / 0.29 ms = 67 TFLOP/s; a library matrix product reaches 150).
//
// Everything is computed transposed (a query per lane), with operands loaded from global memory in MFMA layout: A = a
// row of keys / slots per lane (16 bytes of consecutive columns, four products per load; both operands number the
// contraction the same way, so its order is free), and the accumulator of a score product is the B operand of the next
// product as it stands.  LDS and barriers only where four waves of a unit exchange their parts.  A unit whose output is not
// finite is formed a second time without the rows that a query does not see (f32_out_rows); the look at the output costs
// nothing measurable (567 / 560 us without / with, at B=2, T=4096, 32/8 heads of 128).
#include "common.h"

namespace nha {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int BT = 64;
constexpr int MS = 64;
// A factored decay exp(gc_i - gr) exp(gr - gc_j) with its reference at the start of the 16 rows has one growing factor;
// blocks in which it would pass e^60 take the pairwise form instead.
constexpr float GROWTH_MAX = 60.f;

struct FP {
  const float *q_swa, *k_swa, *q_gsa, *k_gsa, *v, *s, *g;
  float* o;
  float *lse_swa, *lse_gsa;
  const float *h0k, *h0v;
  float *hkt, *hvt;
  const int32_t *cu, *cidx, *coff;
  float* gc;          // [T_tot][H][M]   chunk-local inclusive gate cumsum
  float *hkc, *hvc;   // [NT][H][M][D]   chunk increments, then chunk-start states
  int T_tot, N, NT, HQ, H, NG, wl, shift;
  float scale;
};

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
// e^x to about an ulp: 2^t of the rounded t = x log2(e), corrected to first order for what rounding t lost (an fma recovers
// it exactly).  v_exp_f32 of the rounded product alone is off by |x| 2^-24, the library's expf takes twice the instructions
// for ranges that do not occur here; below e^-200 everything is 0, -inf included.  NaN stays NaN (fmaxf would drop it).
__device__ __forceinline__ float exp_f32(float x) {
  constexpr float HI = 1.44269502f, LO = 1.92596299e-8f, LN2 = 0.693147181f;   // HI + LO = log2(e)
  x = __builtin_elementwise_maximum(x, -200.f);
  const float t = x * HI, lost = fmaf(x, HI, -t) + x * LO, e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, lost * LN2, e);
}
// over the four 16-lane rows of a wave
__device__ __forceinline__ float rows_max(float x) { x = fmaxf(x, __shfl_xor(x, 16, 64)); return fmaxf(x, __shfl_xor(x, 32, 64)); }
__device__ __forceinline__ float rows_sum(float x) { x += __shfl_xor(x, 16, 64); return x + __shfl_xor(x, 32, 64); }

// grid (NT * H, 2): y = 0 the k-state and gc, 1 the v-state.  A wave owns 16 slots: lane (slot l%16, rows 16 (l/16) + i).
template <int D>
__global__ __launch_bounds__(256) void f32_state_local_kernel(const FP p) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, qd = lane >> 4;
  const int m0 = 16 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = m0 + l16;
  const int chunk = blockIdx.x / p.H, h = blockIdx.x % p.H;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int rows = min(BT, eos - bos - it * BT), base = it * BT - p.shift;   // row j absorbs token bos + base + j
  const int jlo = base < 0 ? -base : 0;                                      // first row with a source token
  float g[16], s[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int j = 16 * qd + i, jc = max(min(j, rows - 1), jlo);
    // rows before jlo or from `rows` on absorb nothing; their loads go to a row that exists
    const bool on = j >= jlo && j < rows;
    const int64_t row = jlo < rows ? ((int64_t)(bos + base + jc) * p.H + h) * MS + m : ((int64_t)bos * p.H + h) * MS + m;
    const float gv = p.g[row], sv = p.s[row];
    g[i] = on ? gv : 0.f;
    s[i] = on ? sv : 0.f;
  }
#pragma unroll
  for (int i = 1; i < 16; ++i) g[i] += g[i - 1];
  const float t0 = __shfl(g[15], l16, 64), t1 = __shfl(g[15], 16 + l16, 64), t2 = __shfl(g[15], 32 + l16, 64), t3 = __shfl(g[15], 48 + l16, 64);
  const float before = qd == 0 ? 0.f : qd == 1 ? t0 : qd == 2 ? t0 + t1 : t0 + t1 + t2;
  // A row's decay to the end of the chunk is summed from the gates after it, not taken as a difference of two cumsums that
  // were each rounded at the chunk's whole magnitude: error of the final states against 64 bits at 512 tokens, 4 heads of 64,
  // gates logsigmoid(N(0,1)): 9.3e-7 with the difference, 7.6e-7 in the generic kernels, 1.9e-7 like this.
  const float after = qd == 3 ? 0.f : qd == 2 ? t3 : qd == 1 ? t2 + t3 : t1 + t2 + t3, own = g[15];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    s[i] *= exp_f32(own - g[i] + after);
    const int j = 16 * qd + i;
    if (blockIdx.y == 0 && j < rows) p.gc[((int64_t)(bos + it * BT + j) * p.H + h) * MS + m] = g[i] + before;
  }
  const float* x = blockIdx.y == 0 ? p.k_gsa : p.v;
  float* u = (blockIdx.y == 0 ? p.hkc : p.hvc) + ((int64_t)chunk * p.H + h) * MS * D;
  if (jlo >= rows) {
    for (int c = 0; c < D / 16; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) u[(m0 + 4 * qd + r) * D + 16 * c + l16] = 0.f;
    return;
  }
#pragma unroll 2
  for (int c = 0; c < D / 16; ++c) {
    float b[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int j = max(min(16 * qd + i, rows - 1), jlo);
      b[i] = x[((int64_t)(bos + base + j) * p.H + h) * D + 16 * c + l16];
    }
    if (jlo > 0 || rows < BT)   // rows that absorb nothing: zero, not the row that was read in their place (0 inf is NaN)
#pragma unroll
      for (int i = 0; i < 16; ++i) b[i] = 16 * qd + i >= jlo && 16 * qd + i < rows ? b[i] : 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; ++i) acc = mfma4(s[i], b[i], acc);   // [slot 4 (l/16) + r][column l%16]
#pragma unroll
    for (int r = 0; r < 4; ++r) u[(m0 + 4 * qd + r) * D + 16 * c + l16] = acc[r];
  }
}

// one thread per (sequence, kv-head, state, slot, four columns); loads of eight chunks are requested together
template <int D>
__global__ __launch_bounds__(256) void f32_state_scan_kernel(const FP p) {
  constexpr int Q = D / 4;
  int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int c4 = 4 * (int)(x % Q); x /= Q;
  const int m = (int)(x % MS); x /= MS;
  const bool vs = x % 2; x /= 2;
  const int h = (int)(x % p.H), n = (int)(x / p.H);
  if (n >= p.N) return;
  const int bos = p.cu[n], eos = p.cu[n + 1], c0 = p.coff[n], nc = p.coff[n + 1] - c0;
  const int64_t sh = (int64_t)n * p.H + h;
  f32x4 st = {0.f, 0.f, 0.f, 0.f};
  const float* h0 = vs ? p.h0v : p.h0k;
  if (h0) {
    if (vs) st = ld4(h0 + (sh * MS + m) * D + c4);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) st[e] = h0[(sh * D + c4 + e) * MS + m];
  }
  float* u = (vs ? p.hvc : p.hkc) + (((int64_t)c0 * p.H + h) * MS + m) * D + c4;
  const int64_t step = (int64_t)p.H * MS * D;
  const float* gc = p.gc + (int64_t)h * MS + m;
  for (int c = 0; c < nc; c += 8) {
    f32x4 in[8];
    float gl[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int cc = min(c + e, nc - 1), last = min(bos + (cc + 1) * BT, eos) - 1;
      in[e] = ld4(u + cc * step);
      gl[e] = gc[(int64_t)last * p.H * MS];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (c + e < nc) {
        *reinterpret_cast<f32x4*>(u + (c + e) * step) = st;
        st = st * exp_f32(gl[e]) + in[e];
      }
  }
  if (vs && p.hvt) *reinterpret_cast<f32x4*>(p.hvt + (sh * MS + m) * D + c4) = st;
  if (!vs && p.hkt)
#pragma unroll
    for (int e = 0; e < 4; ++e) p.hkt[(sh * D + c4 + e) * MS + m] = st[e];
}

// 16 rows (block `sub` of a chunk) of one query head.  A product takes its 16 rows of keys, values or strengths for all 16
// queries, the ones that a query does not see (later rows, rows before its window, rows that absorb no token) with weight
// zero: exact for finite values only.  Returns whether an output is not finite, with nothing of the unit settled then;
// EXACT leaves such rows out, query by query and row by row, and always settles it.
template <int D, bool EXACT>
__device__ __forceinline__ bool f32_out_rows(const FP& p, int chunk, int h, int gq, int sub) {
  constexpr int KK = D / 16;   // 16-column pieces of a row
  const int lane = threadIdx.x & 63, l16 = lane & 15, qd = lane >> 4;
  const int hq = h * p.NG + gq;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int cb = bos + it * BT, rows = min(BT, eos - cb);
  if (16 * sub >= rows) return false;
  const int t0 = cb + 16 * sub, t = t0 + l16, tq = min(t, eos - 1);   // the lane's query; rows past the end are not stored
  f32x4 O[KK];
#pragma unroll
  for (int c = 0; c < KK; ++c) O[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
  f32x4 q[KK];
  auto load_q = [&](const float* src) {
#pragma unroll
    for (int c = 0; c < KK; ++c) q[c] = ld4(src + ((int64_t)tq * p.HQ + hq) * D + 16 * c + 4 * qd) * p.scale;
  };
  // S^T[row][query] of 16 rows whose row l%16 starts at x: the loads, the products
  struct Rows { f32x4 a[KK]; };
  auto fetch = [&](const float* x) {
    Rows k;
#pragma unroll
    for (int c = 0; c < KK; ++c) k.a[c] = ld4(x + 16 * c + 4 * qd);
    return k;
  };
  auto scores = [&](const Rows& k) {
    const f32x4* a = k.a;
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KK; ++c)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        acc0 = mfma4(a[c][e], q[c][e], acc0);
        acc1 = mfma4(a[c][e + 1], q[c][e + 1], acc1);
      }
    return acc0 + acc1;
  };
  // O^T += X^T W^T for 16 rows: W in accumulator layout, row(r) = where row 4 (l/16) + r starts
  struct Cols { float a[4][KK]; };
  auto fetch_cols = [&](auto row) {
    Cols v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float* x = row(r) + l16;
#pragma unroll
      for (int c = 0; c < KK; ++c) v.a[r][c] = x[16 * c];
    }
    return v;
  };
  auto read = [&](const Cols& v, const f32x4& w) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < KK; ++c) O[c] = mfma4(v.a[r][c], w[r], O[c]);
  };
  // value of accumulator row jj (of 16) for the lane's query
  auto of_row = [&](const f32x4& w, int jj) { return __shfl(jj & 2 ? (jj & 1 ? w[3] : w[2]) : (jj & 1 ? w[1] : w[0]), 16 * (jj >> 2) + l16, 64); };
  // the same sum over the rows jj that the lane's query sees; row(jj) = where row jj starts
  auto read_seen = [&](auto row, auto seen, const f32x4& w) {
    for (int jj = 0; jj < 16; ++jj) {
      const float x = of_row(w, jj);
      if (!seen(jj)) continue;
#pragma unroll
      for (int c = 0; c < KK; ++c) O[c] += ld4(row(jj) + 16 * c + 4 * qd) * x;
    }
  };

  // ---- window: keys max(bos, t - wl) .. t, newest 16 first (every query meets its own key in the first block) --------
  load_q(p.q_swa);
  const int lo = p.wl < 0 ? bos : max(bos, t0 - p.wl), mylo = p.wl < 0 ? bos : max(bos, t - p.wl);
  float mw = -INFINITY, lw = 0.f;
  auto keys = [&](int kb) { return fetch(p.k_swa + ((int64_t)max(bos, min(kb + l16, eos - 1)) * p.H + h) * D); };
  Rows kr = keys(t0);
  for (int kb = t0; kb > lo - 16; kb -= 16) {
    // the values of this block and the keys of the next are under way while its scores are formed
    auto vrow = [&](int j) { return p.v + ((int64_t)max(bos, min(kb + j, eos - 1)) * p.H + h) * D; };
    Cols vc;
    if constexpr (!EXACT) vc = fetch_cols([&](int r) { return vrow(4 * qd + r); });
    const Rows kn = keys(kb - 16);
    f32x4 s = scores(kr);
    kr = kn;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = kb + 4 * qd + r;
      if (j > tq || j < mylo) s[r] = -INFINITY;
    }
    const float mx = rows_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])));
    const float mn = fmaxf(mw, mx);
    if (__any(mn != mw)) {   // no lane's maximum moved: nothing to rescale
      const float alpha = exp_f32(mw - mn);
      lw *= alpha;
#pragma unroll
      for (int c = 0; c < KK; ++c) O[c] *= alpha;
      mw = mn;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = exp_f32(s[r] - mw);
      lw += s[r];
    }
    if constexpr (EXACT) read_seen(vrow, [&](int jj) { return kb + jj <= tq && kb + jj >= mylo; }, s);
    else read(vc, s);
  }
  lw = rows_sum(lw);

  // ---- slot logits L[m][query], m = 16 b + 4 (l/16) + r -------------------------------------------------------------
  load_q(p.q_gsa);
  const int64_t ch = (int64_t)chunk * p.H + h;
  const float* gcb = p.gc + ((int64_t)cb * p.H + h) * MS;    // gate row of chunk row j: gcb + j * H * MS
  const int gs = p.H * MS;
  const int base = it * BT - p.shift;                         // chunk row j absorbs token bos + base + j
  auto src = [&](int j) { return bos + max(0, min(base + j, eos - bos - 1)); };
  // 1 where row j absorbs a token, else 0: a factor and not a condition, so that the loads it guards need no branch (each
  // branch's loads were waited for on their own)
  auto live = [&](int j) { return base + j >= 0 && j < rows ? 1.f : 0.f; };
  f32x4 gi[4], gr[4], L[4], L2[4];
  float ga[4], growth = 0.f;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    gi[b] = ld4(gcb + (int64_t)(tq - cb) * gs + 16 * b + 4 * qd);
    const int last = min(16 * sub + 15, rows - 1), ref = max(16 * sub - 1, 0);
    gr[b] = sub ? ld4(gcb + (int64_t)ref * gs + 16 * b + 4 * qd) : (f32x4){0.f, 0.f, 0.f, 0.f};
    ga[b] = sub ? gcb[(int64_t)ref * gs + 16 * b + l16] : 0.f;
    growth = fmaxf(growth, ga[b] - gcb[(int64_t)last * gs + 16 * b + l16]);
    L[b] = scores(fetch(p.hkc + (ch * MS + 16 * b + l16) * D));
    L2[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) L[b][r] *= exp_f32(gi[b][r]);
  }
  const bool pairwise = EXACT || __any(growth > GROWTH_MAX);
  f32x4 A;   // intra-chunk scores [row][query] of 16 rows, at last of those of `sub`
  // the logits' share of the 16 rows of J, each with its own decay
  auto add_pairs = [&](int J) {
    for (int jj = 0; jj < 16; ++jj) {
      const int j = 16 * J + jj;
      const float a = of_row(A, jj);
      if (live(j) == 0.f) continue;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const f32x4 sv = ld4(p.s + ((int64_t)src(j) * p.H + h) * MS + 16 * b + 4 * qd), gj = ld4(gcb + (int64_t)j * gs + 16 * b + 4 * qd);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (J < sub || jj <= l16) L[b][r] += a * sv[r] * exp_f32(gi[b][r] - gj[r]);
      }
    }
  };
  for (int J = 0; J <= sub; ++J) {
    if constexpr (EXACT) {
      A = scores(fetch(p.k_gsa + ((int64_t)src(16 * J + l16) * p.H + h) * D));
      add_pairs(J);
      continue;
    }
    float sv[4][4], gv[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * J + 4 * qd + r;
      const float* srow = p.s + ((int64_t)src(j) * p.H + h) * MS + l16;
      const float* grow = gcb + (int64_t)min(j, rows - 1) * gs + l16;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        sv[r][b] = srow[16 * b];
        gv[r][b] = grow[16 * b];
      }
    }
    A = scores(fetch(p.k_gsa + ((int64_t)src(16 * J + l16) * p.H + h) * D));
    if (J == sub) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * qd + r > l16) A[r] = 0.f;
      if (pairwise) break;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * J + 4 * qd + r;
#pragma unroll
      for (int b = 0; b < 4; ++b) L2[b] = mfma4(sv[r][b] * live(j) * exp_f32(ga[b] - gv[r][b]), A[r], L2[b]);
    }
  }
  if constexpr (!EXACT) {
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) L[b][r] += L2[b][r] * exp_f32(gi[b][r] - gr[b][r]);
    if (pairwise) add_pairs(sub);
  }

  // ---- one softmax over [slots | window] ----------------------------------------------------------------------------
  float mg = -INFINITY, lg = 0.f;
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) mg = fmaxf(mg, L[b][r]);
  mg = rows_max(mg);
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      L[b][r] = exp_f32(L[b][r] - mg);
      lg += L[b][r];
    }
  lg = rows_sum(lg);
  if (qd == 0 && t < eos) {
    if (p.lse_gsa) p.lse_gsa[(int64_t)t * p.HQ + hq] = mg + logf(lg);
    if (p.lse_swa) p.lse_swa[(int64_t)t * p.HQ + hq] = mw + logf(lw);
  }
  const float mt = fmaxf(mg, mw), eg = exp_f32(mg - mt), ew = exp_f32(mw - mt);
  const float inv = 1.f / (lg * eg + lw * ew);
#pragma unroll
  for (int c = 0; c < KK; ++c) O[c] *= ew * inv;
#pragma unroll
  for (int b = 0; b < 4; ++b) L[b] *= eg * inv;

  // ---- slot read ----------------------------------------------------------------------------------------------------
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    f32x4 w;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      w[r] = L[b][r] * exp_f32(gi[b][r]);
      L2[b][r] = L[b][r] * exp_f32(gi[b][r] - gr[b][r]);
    }
    read(fetch_cols([&](int r) { return p.hvc + (ch * MS + 16 * b + 4 * qd + r) * D; }), w);
  }
  for (int J = 0; J <= sub; ++J) {
    auto vrow = [&](int j) { return p.v + ((int64_t)src(16 * J + j) * p.H + h) * D; };
    Cols vc;
    if constexpr (!EXACT) vc = fetch_cols([&](int r) { return vrow(4 * qd + r); });
    f32x4 w = {0.f, 0.f, 0.f, 0.f};   // weights [row][query]
    if (!EXACT && (J < sub || !pairwise)) {
      const int j = 16 * J + l16;
      const float* srow = p.s + ((int64_t)src(j) * p.H + h) * MS + 4 * qd;
      const float* grow = gcb + (int64_t)min(j, rows - 1) * gs + 4 * qd;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const f32x4 sv = ld4(srow + 16 * b), gj = ld4(grow + 16 * b);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          w = mfma4(sv[r] * live(j) * exp_f32(gr[b][r] - gj[r]), L2[b][r], w);
        }
      }
    } else {
      for (int jj = 0; jj < 16; ++jj) {
        const int j = 16 * J + jj;
        if (live(j) == 0.f) continue;
        float x = 0.f;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const f32x4 sv = ld4(p.s + ((int64_t)src(j) * p.H + h) * MS + 16 * b + 4 * qd), gj = ld4(gcb + (int64_t)j * gs + 16 * b + 4 * qd);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (J < sub || jj <= l16) x += L[b][r] * sv[r] * exp_f32(gi[b][r] - gj[r]);
        }
        x = rows_sum(x);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (jj == 4 * qd + r) w[r] = x;
      }
    }
    if (J == sub)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * qd + r > l16) w[r] = 0.f;
    if constexpr (EXACT) read_seen(vrow, [&](int jj) { return live(16 * J + jj) != 0.f && (J < sub || jj <= l16); }, w);
    else read(vc, w);
  }
  if constexpr (!EXACT) {
    float z = 0.f;   // NaN if an output is not finite
#pragma unroll
    for (int c = 0; c < KK; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) z = fmaf(O[c][e], 0.f, z);
    if (__any(t < eos && z != 0.f)) return true;
  }
  if (t < eos)
#pragma unroll
    for (int c = 0; c < KK; ++c) *reinterpret_cast<f32x4*>(p.o + ((int64_t)t * p.HQ + hq) * D + 16 * c + 4 * qd) = O[c];
  return false;
}

// (two waves per SIMD up to head size 128: the rare form's registers do not cost the second)
template <int D, int WPB>
__global__ __launch_bounds__(64 * WPB, D <= 128 ? 2 : 1) void f32_out_kernel(const FP p) {
  int unit = blockIdx.x * WPB + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int gq = unit % p.NG; unit /= p.NG;       // the heads of a group and the rows of a chunk share keys: neighbours
  const int sub = unit & 3; unit >>= 2;
  const int h = unit % p.H, chunk = unit / p.H;
  if (chunk >= p.NT) return;
  if (f32_out_rows<D, false>(p, chunk, h, gq, sub)) f32_out_rows<D, true>(p, chunk, h, gq, sub);
}

// The same unit by a workgroup of four waves, for calls with fewer units than the card has room for: a unit alone is one chain
// of dependent loads and products (q, window blocks one after the other, logits, the rows of the chunk twice).  Wave w takes
// every fourth block of window keys and the 16 slots from 16 w on, each with a softmax of its own, and row block w of the
// chunk: its scores for the slots of all waves, and its values with the weights that the four waves' slots give it.  What
// the waves exchange goes through LDS: scores, weights relative to each wave's maximum, at last 3/4 of the outputs.
// Kernel at 512 tokens, 4 heads of 64, W = 64 (128 units): 22.9 -> 12.5 us,
// W = 512 45.0 -> 17.4; 8 heads of 128, W = 64 (256 units) 32.7 -> 16.7; 4 heads of 256 59.5 -> 29.7.  (With the values and
// weights of the slot part requested before the window too: 13.2 and 256 registers, one workgroup per CU.)
template <int D>
__global__ __launch_bounds__(256, D <= 128 ? 2 : 1) void f32_out_split_kernel(const FP p) {
  constexpr int KK = D / 16, OWN = KK / 4;
  constexpr bool EARLY = D == 64;   // the rows of the slot part are under way during the window; wider ones have no room for them
  __shared__ f32x4 lds[12 * OWN > 20 ? 12 * OWN : 20][64];
  __shared__ f32x4 stat[4][16];
  f32x4(*const As)[64] = lds;                                        // [row block][lane]
  f32x4(*const Ws)[4][64] = reinterpret_cast<f32x4(*)[4][64]>(lds + 4);   // [row block][wave][lane]
  f32x4(*const Os)[3][OWN][64] = reinterpret_cast<f32x4(*)[3][OWN][64]>(lds);   // [owner][other wave][piece][lane]
  const int lane = threadIdx.x & 63, l16 = lane & 15, qd = lane >> 4, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int unit = blockIdx.x;
  const int gq = unit % p.NG; unit /= p.NG;
  const int sub = unit & 3; unit >>= 2;
  const int h = unit % p.H, chunk = unit / p.H, hq = h * p.NG + gq;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int cb = bos + it * BT, rows = min(BT, eos - cb);
  if (16 * sub >= rows) return;
  const int t0 = cb + 16 * sub, t = t0 + l16, tq = min(t, eos - 1);
  const int64_t ch = (int64_t)chunk * p.H + h;
  const float* gcb = p.gc + ((int64_t)cb * p.H + h) * MS;
  const int gs = p.H * MS, base = it * BT - p.shift;
  auto src = [&](int j) { return bos + max(0, min(base + j, eos - bos - 1)); };
  auto live = [&](int j) { return base + j >= 0 && j < rows ? 1.f : 0.f; };
  struct Rows { f32x4 a[KK]; };
  struct Cols { float a[4][KK]; };
  auto fetch = [&](const float* x) {
    Rows k;
#pragma unroll
    for (int c = 0; c < KK; ++c) k.a[c] = ld4(x + 16 * c + 4 * qd);
    return k;
  };
  auto fetch_cols = [&](auto row) {
    Cols v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float* x = row(r) + l16;
#pragma unroll
      for (int c = 0; c < KK; ++c) v.a[r][c] = x[16 * c];
    }
    return v;
  };
  auto scores = [&](const Rows& k, const Rows& q) {
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KK; ++c)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        acc0 = mfma4(k.a[c][e], q.a[c][e] * p.scale, acc0);
        acc1 = mfma4(k.a[c][e + 1], q.a[c][e + 1] * p.scale, acc1);
      }
    return acc0 + acc1;
  };
  f32x4 O[KK];
#pragma unroll
  for (int c = 0; c < KK; ++c) O[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto read = [&](const Cols& v, const f32x4& x) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < KK; ++c) O[c] = mfma4(v.a[r][c], x[r], O[c]);
  };
  auto of_row = [&](const f32x4& x, int jj) { return __shfl(jj & 2 ? (jj & 1 ? x[3] : x[2]) : (jj & 1 ? x[1] : x[0]), 16 * (jj >> 2) + l16, 64); };

  // ---- operands ----------------------------------------------------------------------------------------------------
  auto krow = [&](int kb) { return p.k_swa + ((int64_t)max(bos, min(kb + l16, eos - 1)) * p.H + h) * D; };
  const Rows q = fetch(p.q_swa + ((int64_t)tq * p.HQ + hq) * D);
  Rows kr = fetch(krow(t0 - 16 * w));
  Rows qg, hk, kg;
  auto slot_rows = [&] {
    qg = fetch(p.q_gsa + ((int64_t)tq * p.HQ + hq) * D);
    hk = fetch(p.hkc + (ch * MS + 16 * w + l16) * D);
    kg = fetch(p.k_gsa + ((int64_t)src(16 * w + l16) * p.H + h) * D);
  };
  const int last = min(16 * sub + 15, rows - 1), ref = max(16 * sub - 1, 0), m4 = 16 * w + 4 * qd, m1 = 16 * w + l16;
  const f32x4 gi = ld4(gcb + (int64_t)(tq - cb) * gs + m4);
  f32x4 gr = ld4(gcb + (int64_t)ref * gs + m4);
  float ga = gcb[(int64_t)ref * gs + m1];
  const float gl = gcb[(int64_t)last * gs + m1];
  // strengths and gate sums of the chunk's rows: a slot per lane for the logits (here), a row per lane for the weights (later)
  float sa[4][4], gv[4][4];
  f32x4 sw[4], gw[4];
#pragma unroll
  for (int J = 0; J < 4; ++J) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * J + 4 * qd + r;
      sa[J][r] = p.s[((int64_t)src(j) * p.H + h) * MS + m1];
      gv[J][r] = gcb[(int64_t)min(j, rows - 1) * gs + m1];
    }
  }
  if constexpr (EARLY) slot_rows();
  if (!sub) {
    gr = (f32x4){0.f, 0.f, 0.f, 0.f};
    ga = 0.f;
  }

  // ---- window: every fourth block of 16 keys, newest first.  A query may meet no key here: what it does not see counts 0,
  // whatever its maximum --------------------------------------------------------------------------------------------
  const int lo = p.wl < 0 ? bos : max(bos, t0 - p.wl), mylo = p.wl < 0 ? bos : max(bos, t - p.wl);
  float mw = -INFINITY, lw = 0.f;
  for (int kb = t0 - 16 * w; kb > lo - 16; kb -= 64) {
    const Cols vc = fetch_cols([&](int r) { return p.v + ((int64_t)max(bos, min(kb + 4 * qd + r, eos - 1)) * p.H + h) * D; });
    const Rows kn = fetch(krow(kb - 64));
    f32x4 s = scores(kr, q);
    kr = kn;
    float mx = -INFINITY;
    bool seen[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = kb + 4 * qd + r;
      seen[r] = j <= tq && j >= mylo;
      mx = fmaxf(mx, seen[r] ? s[r] : -INFINITY);
    }
    mx = rows_max(mx);
    const float mn = fmaxf(mw, mx);
    if (__any(mn != mw)) {
      const float alpha = mn == mw ? 1.f : exp_f32(mw - mn);
      lw *= alpha;
#pragma unroll
      for (int c = 0; c < KK; ++c) O[c] *= alpha;
      mw = mn;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = seen[r] ? exp_f32(s[r] - mw) : 0.f;
      lw += s[r];
    }
    read(vc, s);
  }
  lw = rows_sum(lw);

  // ---- slot logits L[m][query], m = 16 w + 4 (l/16) + r ------------------------------------------------------------
  if constexpr (!EARLY) slot_rows();
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    const int j = 16 * J + l16;
    sw[J] = ld4(p.s + ((int64_t)src(j) * p.H + h) * MS + m4);
    gw[J] = ld4(gcb + (int64_t)min(j, rows - 1) * gs + m4);
  }
  f32x4 L = scores(hk, qg), L2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < 4; ++r) L[r] *= exp_f32(gi[r]);
  if (w <= sub) {
    f32x4 A = scores(kg, qg);
    if (w == sub)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * qd + r > l16) A[r] = 0.f;
    As[w][lane] = A;
  }
  __syncthreads();
  const bool pairwise = __any(ga - gl > GROWTH_MAX);
  const int fast = pairwise ? sub : sub + 1;   // row blocks whose decays are factored
#pragma unroll
  for (int J = 0; J < 4; ++J)
    if (J < fast) {
      const f32x4 A = As[J][lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) L2 = mfma4(sa[J][r] * live(16 * J + 4 * qd + r) * exp_f32(ga - gv[J][r]), A[r], L2);
    }
#pragma unroll
  for (int r = 0; r < 4; ++r) L[r] += L2[r] * exp_f32(gi[r] - gr[r]);
  auto pair_row = [&](int jj, f32x4* sv, f32x4* gj) {
    const int j = 16 * sub + jj;
    *sv = ld4(p.s + ((int64_t)src(j) * p.H + h) * MS + m4);
    *gj = ld4(gcb + (int64_t)j * gs + m4);
    return live(j) != 0.f;
  };
  if (pairwise) {
    const f32x4 A = As[sub][lane];
    for (int jj = 0; jj < rows - 16 * sub && jj < 16; ++jj) {
      const float a = of_row(A, jj);
      f32x4 sv, gj;
      if (!pair_row(jj, &sv, &gj)) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (jj <= l16) L[r] += a * sv[r] * exp_f32(gi[r] - gj[r]);
    }
  }

  // ---- softmax over this wave's slots and keys, its slots' read, the weights that its slots give the chunk's rows ------
  float mg = rows_max(fmaxf(fmaxf(L[0], L[1]), fmaxf(L[2], L[3]))), lg = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    L[r] = exp_f32(L[r] - mg);
    lg += L[r];
  }
  lg = rows_sum(lg);
  const float mt = fmaxf(mg, mw), eg = exp_f32(mg - mt), ew = exp_f32(mw - mt);
#pragma unroll
  for (int c = 0; c < KK; ++c) O[c] *= ew;
  f32x4 wr;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    L[r] *= eg;
    wr[r] = L[r] * exp_f32(gi[r]);
    L2[r] = L[r] * exp_f32(gi[r] - gr[r]);
  }
#pragma unroll
  for (int J = 0; J < 4; ++J)
    if (J < fast) {
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) x = mfma4(sw[J][r] * live(16 * J + l16) * exp_f32(gr[r] - gw[J][r]), L2[r], x);
      Ws[J][w][lane] = x;
    }
  if (pairwise) {
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    for (int jj = 0; jj < rows - 16 * sub && jj < 16; ++jj) {
      f32x4 sv, gj;
      if (!pair_row(jj, &sv, &gj)) continue;
      float y = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (jj <= l16) y += L[r] * sv[r] * exp_f32(gi[r] - gj[r]);
      y = rows_sum(y);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (jj == 4 * qd + r) x[r] = y;
    }
    Ws[sub][w][lane] = x;
  }
  if (qd == 0) stat[w][l16] = (f32x4){mw, lw, mg, lg};
  read(fetch_cols([&](int r) { return p.hvc + (ch * MS + 16 * w + 4 * qd + r) * D; }), wr);
  const Cols vj = fetch_cols([&](int r) { return p.v + ((int64_t)src(16 * w + 4 * qd + r) * p.H + h) * D; });
  __syncthreads();

  // ---- the four softmaxes as one -----------------------------------------------------------------------------------
  f32x4 st[4];
  float MW = -INFINITY, LW = 0.f, MG = -INFINITY, LG = 0.f;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    st[x] = stat[x][l16];
    MW = fmaxf(MW, st[x][0]);
    MG = fmaxf(MG, st[x][2]);
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    LW += st[x][1] * exp_f32(st[x][0] - MW);
    LG += st[x][3] * exp_f32(st[x][2] - MG);
  }
  const float MT = fmaxf(MG, MW), inv = 1.f / (LG * exp_f32(MG - MT) + LW * exp_f32(MW - MT));
  float part[4];   // wave x's outputs and weights are relative to its own maximum
#pragma unroll
  for (int x = 0; x < 4; ++x) part[x] = exp_f32(fmaxf(st[x][2], st[x][0]) - MT) * inv;
  const float mine = exp_f32(mt - MT) * inv;
#pragma unroll
  for (int c = 0; c < KK; ++c) O[c] *= mine;
  if (w <= sub) {
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int y = 0; y < 4; ++y) x += Ws[w][y][lane] * part[y];
    if (w == sub)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * qd + r > l16) x[r] = 0.f;
    read(vj, x);
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < KK; ++c)   // (unrolled over all pieces: O is indexed by constants only)
    if (c / OWN != w) Os[c / OWN][(w - c / OWN - 1) & 3][c % OWN][lane] = O[c];
  __syncthreads();
  f32x4 out[OWN];
#pragma unroll
  for (int c = 0; c < KK; ++c)
    if (c / OWN == w) out[c % OWN] = O[c];
  float z = 0.f;   // NaN if an output is not finite
#pragma unroll
  for (int c = 0; c < OWN; ++c) {
    out[c] += Os[w][0][c][lane] + Os[w][1][c][lane] + Os[w][2][c][lane];
#pragma unroll
    for (int e = 0; e < 4; ++e) z = fmaf(out[c][e], 0.f, z);
  }
  if (__syncthreads_or(t < eos && z != 0.f)) {
    if (w == 0) f32_out_rows<D, true>(p, chunk, h, gq, sub);
    return;
  }
  if (t >= eos) return;
  if (w == 0 && qd == 0) {
    if (p.lse_gsa) p.lse_gsa[(int64_t)t * p.HQ + hq] = MG + logf(LG);
    if (p.lse_swa) p.lse_swa[(int64_t)t * p.HQ + hq] = MW + logf(LW);
  }
#pragma unroll
  for (int c = 0; c < OWN; ++c) *reinterpret_cast<f32x4*>(p.o + ((int64_t)t * p.HQ + hq) * D + 16 * (w * OWN + c) + 4 * qd) = out[c];
}

template <int D>
int run(const FP& p, int phase, hipStream_t st) {
  if (phase != 2) {
    hipLaunchKernelGGL((f32_state_local_kernel<D>), dim3(p.NT * p.H, 2), dim3(256), 0, st, p);
    const int64_t threads = (int64_t)p.N * p.H * 2 * MS * (D / 4);
    hipLaunchKernelGGL((f32_state_scan_kernel<D>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, p);
    NHA_CHECK_LAUNCH("nha_prefill_fwd(fp32 state pass)");
  }
  if (phase != 1) {
    // Workgroups of four waves (neighbouring units share keys through L1) once there are four per CU, of one wave before.
    const int64_t units = (int64_t)p.NT * p.H * 4 * p.NG;
    // Four waves per unit up to two such workgroups per CU (kernel, a wave / four waves per unit): W = 64, 32 units 22.8 / 12.3,
    // 256 units 23.8 / 12.8, 512 units 26.4 / 20.7, 1024 units 28.1 / 36.0 us (heads of 64); 512 units of 128 36.6 / 26.8,
    // 1024 42.5 / 49.2; 512 of 256 68.7 / 63.8, 1024 72.8 / 120.9.  The rows of the chunk and their decays are worked off once
    // more per wave, so the split costs where the CUs are full anyway.
    if (units <= 512) hipLaunchKernelGGL((f32_out_split_kernel<D>), dim3((unsigned)units), dim3(256), 0, st, p);
    else if (units >= 1024) hipLaunchKernelGGL((f32_out_kernel<D, 4>), dim3((unsigned)((units + 3) / 4)), dim3(256), 0, st, p);
    else hipLaunchKernelGGL((f32_out_kernel<D, 1>), dim3((unsigned)units), dim3(64), 0, st, p);
    NHA_CHECK_LAUNCH("nha_prefill_fwd(fp32 output pass)");
  }
  return NHA_OK;
}

size_t aligned(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace

// Rows are read and written 16 bytes at a time; tensors that start elsewhere (a view into a buffer) keep the generic kernels,
// which read single floats there.
bool prefill_f32_supported(const NhaPrefillArgs* a) {
  uintptr_t at = 0;
  for (const void* x : {a->q_swa, a->k_swa, a->q_gsa, a->k_gsa, a->v, a->s, (const void*)a->o, (const void*)a->h0v, (const void*)a->hvt, (const void*)a->scratch})
    at |= reinterpret_cast<uintptr_t>(x);
  return (at & 15) == 0 && a->dtype == NHA_DTYPE_F32 && a->K == a->V && (a->K == 64 || a->K == 128 || a->K == 256) && a->M == MS &&
         (int64_t)a->NT * a->H * 4 * (a->HQ / a->H) < ((int64_t)1 << 31);
}

// the scratch is that of prefill_simple.hip: gc | k-states | v-states
int prefill_f32_impl(const NhaPrefillArgs* a, int phase) {
  FP p;
  p.q_swa = (const float*)a->q_swa; p.k_swa = (const float*)a->k_swa; p.q_gsa = (const float*)a->q_gsa; p.k_gsa = (const float*)a->k_gsa;
  p.v = (const float*)a->v; p.s = (const float*)a->s; p.g = (const float*)a->g; p.o = (float*)a->o;
  p.lse_swa = a->lse_swa; p.lse_gsa = a->lse_gsa;
  p.h0k = a->h0k; p.h0v = a->h0v; p.hkt = a->hkt; p.hvt = a->hvt;
  p.cu = a->cu_seqlens; p.cidx = a->chunk_indices; p.coff = a->chunk_offsets;
  char* sc = (char*)a->scratch;
  p.gc = (float*)sc;
  sc += aligned((size_t)a->T_tot * a->H * a->M * 4);
  p.hkc = (float*)sc;
  sc += aligned((size_t)a->NT * a->H * a->K * a->M * 4);
  p.hvc = (float*)sc;
  p.T_tot = a->T_tot; p.N = a->N; p.NT = a->NT; p.HQ = a->HQ; p.H = a->H; p.NG = a->HQ / a->H;
  p.wl = a->wl; p.shift = a->shift; p.scale = a->scale;
  hipStream_t st = (hipStream_t)a->stream;
  if (a->K == 64) return run<64>(p, phase, st);
  if (a->K == 128) return run<128>(p, phase, st);
  return run<256>(p, phase, st);
}

}  // namespace nha
