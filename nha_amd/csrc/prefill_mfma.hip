// bf16 MFMA prefill for gfx950 (K == V == D in {64,128,256}, M == 64 slots), fp32 accumulation.
//
// Everything is computed "transposed" so that each lane owns ONE query column of a 16x16
// accumulator block (v_mfma_f32_16x16x32_bf16: A[i][8*(l/16)+e], B[8*(l/16)+e][j], C[4*(l/16)+r][l%16]):
//   S^T[key][q]  = K  Q^T      A = K rows from LDS (16-byte reads), B = Q fragments kept in registers
//   O^T[d][q]   += V^T P^T     A = V^T via ds_read_b64_tr_b16 on the row-major V tile, B = P from the
//                              accumulator layout of S^T directly (contraction index permuted the same
//                              way on both operands), so P never moves between lanes
// Row statistics of the online softmax are per-lane scalars (+2 cross-lane steps over l/16).
// The slot branch is folded into the same machinery: slot logits are an "S tile" against the
// transposed chunk-start state hkT[m][d] and the slot read is a "PV tile" against hv[m][v]; the
// intra-chunk terms use the chunk algebra of nha_fla/ops/nha/chunk_fused.py:186-222, :242-275 with
// 16-row sub-blocks and sub-block-start decay references (:182-184, :203-204).
//
//   state pass  (mfma_state_kernel): per (sequence, kv-head, 16-slot block) sweep over 64-row chunks
//               with the fp32 state held in MFMA accumulators (chunk_fused.py:30-113).
//   output pass (mfma_out_kernel)  : per (chunk, kv-head, group of <=4 q-heads).
#include "prefill_exact.h"

#include <mutex>
#include <stdlib.h>

namespace nha {
namespace {

using namespace mf;

// ------------------------------------------------------------------------------------------
// cooperative 64-row tile copy, global -> registers -> LDS (16-byte pieces, zero fill)
// ------------------------------------------------------------------------------------------
template <int ROWS, int D, int NTHR>
struct TileRegs {
  uint4 r[ROWS * D / 8 / NTHR];
};

// rows of the tile map to global rows grow0 + j; rows outside [vlo, vhi) are zero
template <int ROWS, int D, int NTHR>
__device__ __forceinline__ void tile_g2r(TileRegs<ROWS, D, NTHR>& t, const bf16_t* base, int64_t row_stride,
                                         int64_t grow0, int vlo, int vhi, int tid) {
#pragma unroll
  for (int u = 0; u < ROWS * D / 8 / NTHR; ++u) {
    const int c = tid + NTHR * u;
    const int row = c / (D / 8), col = (c % (D / 8)) * 8;
    uint4 x = make_uint4(0, 0, 0, 0);
    if (row >= vlo && row < vhi) x = *reinterpret_cast<const uint4*>(base + (grow0 + row) * row_stride + col);
    t.r[u] = x;
  }
}
template <int ROWS, int D, int NTHR>
__device__ __forceinline__ void tile_r2l(lbf16* lds, const TileRegs<ROWS, D, NTHR>& t, int tid) {
#pragma unroll
  for (int u = 0; u < ROWS * D / 8 / NTHR; ++u) {
    const int c = tid + NTHR * u;
    const int row = c / (D / 8), col = (c % (D / 8)) * 8;
    lds_st16(lds + row * (D + 16) + col, t.r[u]);
  }
}

// ==========================================================================================
// state pass, two levels
// ==========================================================================================
// The slot recurrence is sequential over the chunks of a sequence, so it is cut into segments of
// 1, 2, 4 or SEG = 8 chunks (plan_scratch).  Level 1 (mfma_state_local_kernel, one workgroup per (segment, kv-head), one wave
// per 16-slot block) runs the recurrence of chunk_fused.py:30-113 from a ZERO state over its
// segment and stores, per chunk, the local chunk-start states, the gate cumsum table and the
// decay accumulated since the segment start; per segment, the local end state and total decay.
// Level 2 carries the true state across segments element-wise, h_seg[s+1] = h_seg[s] * dtot[s] + hend[s],
// in one of two forms.  The forward turns every chunk-start state into the true one, h_loc + h_seg * dcum,
// rounded to bf16 in place, so that the output pass reads plain operand tiles (state_link_kernel, or
// state_scan_kernel followed by state_apply_kernel).  The backward (state_scan_kernel) keeps the
// segment-local states and writes the segment-start states h_seg beside them: it needs the sum in fp32.
// Both states are kept as C[d][m] accumulators (slot m = lane % 16).

// DW: columns of the state one workgroup carries (D, or D/2: twice the workgroups with half the
// tile, which this latency-bound kernel turns into bandwidth; the gates are then read once more).
template <int D> constexpr int LOCAL_DW = D >= 256 ? D / 2 : D;   // measured: 96 -> 88 us at B=8 T=2048 H=4 D=256; no gain at D = 128

// What state_link_kernel may not leave out although the decays after it multiply to zero: initial and end states that are not finite, or not
// far below fp32's limit, and segments that grow.  A word per (segment slot, kv-head, state and column range of level 1, 16 slots), where
// the scan, if it follows instead, leaves its segment-start states.
__device__ __forceinline__ unsigned magnitude(float x) { return __float_as_uint(x) & 0x7fffffffu; }   // (NaNs count too: this file is built without them)
constexpr unsigned ODD_STATE = 0x5f800000u;   // 2^64
__device__ __forceinline__ int* odd_words(const MP& p) { return (int*)p.hseg_k; }

template <int D, int DW>
__global__ __launch_bounds__(256) void mfma_state_local_kernel(const MP p) {
  constexpr int LDT = DW + 16;
  constexpr int NB = DW / 16;
  extern __shared__ __align__(16) unsigned char smem[];
  lbf16* Xt = (lbf16*)smem;
  lbf16* St = Xt + BT * LDT;
  lbf16* Gt = St + BT * SLD;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, kb = lane >> 4;
  const int H = p.H;
  // One-dimensional grid, blockIdx.x = (state and column range z, kv-head h) + H Z k with k counting the segments of
  // the call one sequence after the other, without gaps: the workgroups that find k past the last segment (the grid
  // is sized for the most segments NT chunks in N sequences can have) are the last of the launch.  A workgroup
  // holds its CU slot for the whole chain of its segment and two fit a CU: were workgroups that leave at once
  // strewn over the launch order, the shader engines' shares of the working ones would differ, some CUs would
  // get a third one after their first two and others only one -- a second round for a tenth of the chip (49 us
  // against 32 us per launch at 512 segments x heads x states on 256 CUs).
  // z picks the state: even = k-state (rows of k_gsa; it also writes the gate tables), odd = v-state (rows of v).
  // The two recurrences share nothing but the gates, and twice the workgroups of half the size fill the chip better.
  constexpr int Z = 2 * (D / DW);
  const int hz = blockIdx.x % (H * Z), k = blockIdx.x / (H * Z);
  const int h = hz % H, z = hz / H;
  const bool isv = (z & 1) != 0;
  const int dcol0 = (z >> 1) * DW;             // first state column of this workgroup
  const bool lead = dcol0 == 0;                // writes what does not depend on the column range
  const bf16_t* xsrc = (isv ? p.v : p.k_gsa) + dcol0;
  bf16_t* hloc = isv ? p.hvc : p.hkT;
  float* hend = isv ? p.hend_v : p.hend_k;
  // segment k of the call -> (sequence n, segment kseg of it): a running count of ceil(chunks / segment) over the
  // sequences, 256 at a time (one per thread, prefix over the workgroup)
  __shared__ int seg_wave[4], seg_hit[2];
  int n = 0, kseg = 0;
  {
    int base = 0;
    for (int n0 = 0; n0 < p.N; n0 += 256) {
      const int i = n0 + tid;
      const int segs = i < p.N ? (p.coff[i + 1] - p.coff[i] + (1 << p.seg_sh) - 1) >> p.seg_sh : 0;
      int incl = segs;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o, 64);
        if (lane >= o) incl += t;
      }
      if (lane == 63) seg_wave[wave] = incl;
      __syncthreads();
      int before = base;
      for (int w = 0; w < wave; ++w) before += seg_wave[w];
      const int first = before + incl - segs;
      if (k >= first && k < first + segs) {
        seg_hit[0] = i;
        seg_hit[1] = k - first;
      }
      base += seg_wave[0] + seg_wave[1] + seg_wave[2] + seg_wave[3];
      __syncthreads();
      if (k < base) break;
    }
    if (k >= base) return;   // past the last segment of the call
    n = seg_hit[0];
    kseg = seg_hit[1];
  }
  const int it0 = kseg << p.seg_sh;
  const int chunk0 = p.coff[n] + it0;
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int L = eos - bos;
  const int nchunks = (L + BT - 1) / BT;
  const int nloc = (nchunks - it0) < (1 << p.seg_sh) ? (nchunks - it0) : 1 << p.seg_sh;
  const int m = wave * 16 + l16;   // this lane's slot

  f32x4 hx[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) hx[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float gsum = 0.f;   // sum of the chunk-end gate cumsums since the segment start, this lane's slot

  TileRegs<BT, DW, 256> rx;
  uint4 rs[2], rg[2];
  auto issue = [&](int it) {
    const int rows = (L - it * BT) < BT ? (L - it * BT) : BT;
    const int64_t grow0 = (int64_t)bos + it * BT - p.shift;
    int vlo = p.shift - it * BT;
    vlo = vlo < 0 ? 0 : vlo;
    tile_g2r<BT, DW, 256>(rx, xsrc + (int64_t)h * D, (int64_t)H * D, grow0, vlo, rows, tid);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c8 = tid + 256 * u;
      const int j = c8 >> 3, m8 = (c8 & 7) * 8;
      uint4 xs = make_uint4(0, 0, 0, 0), xg = xs;
      if (j >= vlo && j < rows) {
        xs = *reinterpret_cast<const uint4*>(p.s + ((grow0 + j) * H + h) * MS + m8);
        xg = *reinterpret_cast<const uint4*>(p.g + ((grow0 + j) * H + h) * MS + m8);
      }
      rs[u] = xs;
      rg[u] = xg;
    }
  };

  issue(it0);
  for (int jc = 0; jc < nloc; ++jc) {
    const int it = it0 + jc;
    const int chunk = chunk0 + jc;
    const int rows = (L - it * BT) < BT ? (L - it * BT) : BT;
    if (jc > 0) __syncthreads();   // everyone is done reading the previous chunk's tiles
    tile_r2l<BT, DW, 256>(Xt, rx, tid);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c8 = tid + 256 * u;
      const int j = c8 >> 3, m8 = (c8 & 7) * 8;
      lds_st16(St + j * SLD + m8, rs[u]);
      lds_st16(Gt + j * SLD + m8, rg[u]);
    }
    if (jc + 1 < nloc) issue(it + 1);
    __syncthreads();
    // this lane's rows: element e = 4*q + r is row t = 16*q + 4*kb + r
    // (the sixteen gate and s values of a lane are a column of their tiles: four transposing reads each
    // instead of sixteen 2-byte reads)
    float gcv[16], sg[16];
    const bf16x8 gq01 = lds_frag_tr(Gt, SLD, 0, 16, 16 * wave, lane), gq23 = lds_frag_tr(Gt, SLD, 32, 48, 16 * wave, lane);
    const bf16x8 sq01 = lds_frag_tr(St, SLD, 0, 16, 16 * wave, lane), sq23 = lds_frag_tr(St, SLD, 32, 48, 16 * wave, lane);
    // the chunk's last cumsum: rows without a source token and past the end have gate 0, so it is the sum of all
    float glast = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float a = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        a += (float)(q < 2 ? gq01[4 * q + r] : gq23[4 * (q - 2) + r]);
        gcv[4 * q + r] = a;
      }
      // the sums of the four 16-lane rows, for every lane (lane swaps: sixteen LDS permutes took 1.3k of a chunk's 7.7k cycles)
      const unsigned u = __float_as_uint(a);
      const auto x = __builtin_amdgcn_permlane16_swap(u, u, false, false);
      const auto y0 = __builtin_amdgcn_permlane32_swap(x[0], x[0], false, false), y1 = __builtin_amdgcn_permlane32_swap(x[1], x[1], false, false);
      const float row[4] = {__uint_as_float(y0[0]), __uint_as_float(y1[0]), __uint_as_float(y0[1]), __uint_as_float(y1[1])};
      float off = glast;
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) {
        if (k2 < kb) off += row[k2];
        glast += row[k2];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) gcv[4 * q + r] += off;
    }
    const int64_t cg = (int64_t)chunk * H + h;
    if (lead) {
      // the gate table: rows 0..31 from the k-state workgroup, rows 32..63 from the v-state one (both hold it)
      float* gout = p.gc + cg * BT * MS + m;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int ee = isv ? e + 8 : e;
        gout[(16 * (ee >> 2) + 4 * kb + (ee & 3)) * MS] = isv ? gcv[e + 8] : gcv[e];
      }
    }
    if (!isv && lead) {
      if (kb == 0) p.dcum[cg * MS + m] = fexp(gsum);
      // 16-row sub-blocks over which some slot decays by more than exp(DECAY_CLAMP): the output
      // pass cannot factor their intra-block decay, and their rows are formed again exactly (prefill_exact.h)
      int bits = 0;
      if (kb == 3) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float ref = q > 0 ? gcv[4 * q - 1] : 0.f;
          if (ref - gcv[4 * q + 3] > DECAY_CLAMP) bits |= 1 << q;
        }
      }
#pragma unroll
      for (int x = 32; x >= 1; x >>= 1) bits |= __shfl_xor(bits, x, 64);
      if (lane == 0) p.flags[cg * 4 + wave] = bits;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int t = 16 * (e >> 2) + 4 * kb + (e & 3);
      sg[e] = (t < rows) ? (float)(e < 8 ? sq01[e] : sq23[e - 8]) * fexp(glast - gcv[e]) : 0.f;
    }
    bf16x8 sg0, sg1;   // contraction steps over rows [0,32) and [32,64)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sg0[e] = (__bf16)sg[e];
      sg1[e] = (__bf16)sg[8 + e];
    }
    // local chunk-start states (bf16), before the update: rows m.  A lane holds 4 consecutive d of every 16-column
    // block; the lanes of an even 16-lane row keep block b, those of the odd row block b + 1, and the two trade their
    // halves, so that a lane stores 16 bytes and a row of the state 64 consecutive bytes per instruction
#pragma unroll
    for (int b = 0; b < NB; b += 2) {
      bf16x4 pa, pb;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pa[r] = (__bf16)hx[b][r];
        pb[r] = (__bf16)hx[b + 1][r];
      }
      uint2 ua = __builtin_bit_cast(uint2, pa), ub = __builtin_bit_cast(uint2, pb);
      const auto s0 = __builtin_amdgcn_permlane16_swap(ua.x, ub.x, false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(ua.y, ub.y, false, false);
      const int dcol = 16 * (b + (kb & 1)) + 8 * (kb >> 1);
      *reinterpret_cast<uint4*>(hloc + (cg * MS + m) * D + dcol0 + dcol) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
    }
    const float dk = fexp(glast);
    gsum += glast;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int r = 0; r < 4; ++r) hx[b][r] *= dk;
      // h[d][m] += sum_t x[t][d] sg[t][m]     A = x^T (transposed LDS read), B = sg
      hx[b] = mfma16(lds_frag_tr(Xt, LDT, 0, 16, 16 * b, lane), sg0, hx[b]);
      hx[b] = mfma16(lds_frag_tr(Xt, LDT, 32, 48, 16 * b, lane), sg1, hx[b]);
    }
  }
  // the initial state's part of the first segment's word: this wave's 16 slots and the workgroup's columns of it
  unsigned most = 0;
  if (kseg == 0 && p.h0k) {
    const int64_t nh = (int64_t)n * H + h;
    const float* const src = isv ? p.h0v + (nh * MS + 16 * wave) * D + dcol0 : p.h0k + (nh * D + dcol0) * MS + 16 * wave;
    constexpr int VL = DW / 4;   // lanes to a row of the v-state
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int e = lane + 64 * i;
      const float4 x = *reinterpret_cast<const float4*>(src + (isv ? e / VL * D + e % VL * 4 : e / 4 * MS + e % 4 * 4));
      most = max(most, max(max(magnitude(x.x), magnitude(x.y)), max(magnitude(x.z), magnitude(x.w))));
    }
  }
  // segment end: local state (fp32, [m][d]) and total decay
  const int64_t sl = (int64_t)seg_slot(p.coff, n, it0, p.seg_sh) * H + h;
#pragma unroll
  for (int b = 0; b < NB; ++b)
    *reinterpret_cast<float4*>(hend + (sl * MS + m) * D + dcol0 + 16 * b + 4 * kb) = make_float4(hx[b][0], hx[b][1], hx[b][2], hx[b][3]);
  const float dt = fexp(gsum);
  if (kb == 0 && !isv && lead) p.dtot[sl * MS + m] = dt;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) most = max(most, magnitude(hx[b][r]));
  const int odd = __any(most >= ODD_STATE || magnitude(dt) > __float_as_uint(1.f));
  if (lane == 0) odd_words(p)[(sl * Z + z) * 4 + wave] = odd;
}

// Level 2, the scan: four consecutive d of one slot per thread, sequential over the segments of its sequence;
// writes the true segment-start states h_seg and the final states.  The loads do not depend on the chain, so the
// end states and decays of SCAN_AHEAD segments are requested together, one group ahead of the group that is
// being combined: a thread waits for memory once per group, not once per segment.
// grid (N*H, 2*MS*D/1024): the first MS*D/4 groups are the k-state ([m][d]), the rest the v-state.
constexpr int SCAN_AHEAD = 4;
constexpr int LINK_SEGS = 16;   // average segments of a sequence up to which the forward takes state_link_kernel instead

// What a workgroup of level 2 owns: 16 slots x 64 columns of one state, a slot and four consecutive columns per thread (256
// consecutive bytes of a row of the scratch's [m][d] states per 16 threads).  The caller's k-states lie [d][m]: they pass through
// LDS, 16 slots (64 bytes) of a row side by side.  With a thread's own four columns read and written there one by one, level 2 of a call
// with initial and final states was bound by that (16 packed sequences, 4 heads of 256, 32768 tokens:
// state_scan_kernel 31 -> 23 us).
template <int D>
struct StatePart {
  static constexpr int GROUPS = MS * D / 1024;   // workgroups per state
  bool isv;
  int m, d;
  __device__ __forceinline__ StatePart(int group, int tid) {
    isv = group >= GROUPS;
    const int g = isv ? group - GROUPS : group;
    m = 16 * (g / (D / 64)) + (tid >> 4);
    d = 64 * (g % (D / 64)) + 4 * (tid & 15);
  }
  // tr: [64 d][17] floats of the workgroup; k: the sequence and head's [D][MS]
  __device__ __forceinline__ float4 load_k(const float* k, lfloat* tr, int tid) const {
    const int m0 = m & ~15, d0 = d & ~63;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int x = (tid >> 4) + 16 * i;
      tr[x * 17 + (tid & 15)] = k[(d0 + x) * MS + m0 + (tid & 15)];
    }
    __syncthreads();
    const lfloat* const t = tr + (d & 63) * 17 + (m & 15);
    return make_float4(t[0], t[17], t[34], t[51]);
  }
  __device__ __forceinline__ void store_k(float* k, const float4& v, lfloat* tr, int tid) const {
    const int m0 = m & ~15, d0 = d & ~63;
    lfloat* const t = tr + (d & 63) * 17 + (m & 15);
    __syncthreads();
    t[0] = v.x; t[17] = v.y; t[34] = v.z; t[51] = v.w;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int x = (tid >> 4) + 16 * i;
      k[(d0 + x) * MS + m0 + (tid & 15)] = tr[x * 17 + (tid & 15)];
    }
  }
};

template <int D>
__global__ __launch_bounds__(256) void state_scan_kernel(const MP p) {
  __shared__ float trs[64 * 17];
  lfloat* const tr = (lfloat*)trs;
  const int H = p.H;
  const int n = blockIdx.x / H, h = blockIdx.x % H;
  const StatePart<D> part(blockIdx.y, threadIdx.x);
  const bool isv = part.isv;
  const int m = part.m, d = part.d;
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int nchunks = (eos - bos + BT - 1) / BT;
  const int nseg = (nchunks + (1 << p.seg_sh) - 1) >> p.seg_sh;
  const int64_t nh = (int64_t)n * H + h;
  float4 hcur = make_float4(0.f, 0.f, 0.f, 0.f);
  if (p.h0k) hcur = isv ? *reinterpret_cast<const float4*>(p.h0v + (nh * MS + m) * D + d) : part.load_k(p.h0k + nh * D * MS, tr, threadIdx.x);
  const float* __restrict__ hend = isv ? p.hend_v : p.hend_k;
  float* __restrict__ hseg = isv ? p.hseg_v : p.hseg_k;
  const float* __restrict__ dtot = p.dtot;
  const int slot0 = (p.coff[n] >> p.seg_sh) + n;
  struct Grp {
    float4 he[SCAN_AHEAD];
    float dt[SCAN_AHEAD];
  };
  auto request = [&](Grp& g, int sg0) {
#pragma unroll
    for (int i = 0; i < SCAN_AHEAD; ++i) {
      g.he[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      g.dt[i] = 0.f;
      if (sg0 + i < nseg) {
        const int64_t sl = (int64_t)(slot0 + sg0 + i) * H + h;
        g.he[i] = *reinterpret_cast<const float4*>(hend + (sl * MS + m) * D + d);
        g.dt[i] = dtot[sl * MS + m];
      }
    }
  };
  Grp cur, nxt;
  request(cur, 0);
  for (int sg0 = 0; sg0 < nseg; sg0 += SCAN_AHEAD) {
    if (sg0 + SCAN_AHEAD < nseg) request(nxt, sg0 + SCAN_AHEAD);
#pragma unroll
    for (int i = 0; i < SCAN_AHEAD; ++i) {
      if (sg0 + i < nseg) {
        const int64_t sl = (int64_t)(slot0 + sg0 + i) * H + h;
        *reinterpret_cast<float4*>(hseg + (sl * MS + m) * D + d) = hcur;
        hcur.x = hcur.x * cur.dt[i] + cur.he[i].x;
        hcur.y = hcur.y * cur.dt[i] + cur.he[i].y;
        hcur.z = hcur.z * cur.dt[i] + cur.he[i].z;
        hcur.w = hcur.w * cur.dt[i] + cur.he[i].w;
      }
    }
    cur = nxt;
  }
  if (p.hkt) {
    if (isv) *reinterpret_cast<float4*>(p.hvt + (nh * MS + m) * D + d) = hcur;
    else part.store_k(p.hkt + nh * D * MS, hcur, tr, threadIdx.x);
  }
}

// Level 2, forward form: every chunk-start state becomes the true one, h_loc + h_seg * dcum, rounded to bf16 in
// place, so that the output pass reads plain operand tiles.
//
// Where the carried part h_seg * dcum is below CARRY_FLOOR in absolute value for all four elements of a thread,
// the local state is left as it is -- neither read nor written: the sum would be the local state again to within
// 2^-100, fifty binary orders below anything bf16 tensors of representable magnitude can show.  Gates that forget
// quickly (log-gates of about -1 per token: e^-80 per chunk) leave only the first chunk of a segment to rewrite;
// with slow gates (the layers' logsigmoid / 8: e^-5 per chunk) every chunk is rewritten.
//
// Two forms.  state_link_kernel forms the state that enters a segment itself, from the end states of the segments before it: for
// sequences of up to LINK_SEGS segments.  state_apply_kernel runs after state_scan_kernel, which hands that state on through memory.
constexpr float CARRY_FLOOR = 0x1p-100f;

// What a thread of either form does: four consecutive d of a slot in every chunk of a segment
struct Rewrite {
  uint2 loc[SEG];
  float dc[SEG];
  unsigned need;
  __device__ __forceinline__ void request_decays(const float* dcum, int64_t step, int nloc) {
#pragma unroll
    for (int jc = 0; jc < SEG; ++jc) dc[jc] = jc < nloc ? dcum[(int64_t)jc * step] : 0.f;
  }
  // hloc: the thread's place in the first chunk, step elements before that of the next
  __device__ __forceinline__ void request(const bf16_t* hloc, int64_t step, float amax) {
    need = 0;
#pragma unroll
    for (int jc = 0; jc < SEG; ++jc) {
      loc[jc] = make_uint2(0, 0);
      if (amax * dc[jc] >= CARRY_FLOOR) {
        need |= 1u << jc;
        loc[jc] = *reinterpret_cast<const uint2*>(hloc + jc * step);
      }
    }
  }
  __device__ __forceinline__ void store(bf16_t* hloc, int64_t step, const float (&hs)[4]) const {
#pragma unroll
    for (int jc = 0; jc < SEG; ++jc) {
      if (need & (1u << jc)) {
        const uint32_t w[2] = {loc[jc].x, loc[jc].y};
        bf16x4 o4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float a0 = __uint_as_float((i & 1) ? (w[i >> 1] & 0xffff0000u) : (w[i >> 1] << 16));
          o4[i] = (__bf16)(a0 + hs[i] * dc[jc]);
        }
        *reinterpret_cast<bf16x4*>(hloc + jc * step) = o4;
      }
    }
  }
};

// (sequence, first chunk) of a segment slot (seg_slot)
__device__ __forceinline__ void segment_of(const MP& p, int slot, int& n, int& it0) {
  int lo = 0, hi = p.N - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((p.coff[mid] >> p.seg_sh) + mid <= slot) lo = mid; else hi = mid - 1;
  }
  n = lo;
  it0 = (slot - ((p.coff[n] >> p.seg_sh) + n)) << p.seg_sh;
}

// One launch instead of scan and rewrite: four consecutive d of one slot per thread, every segment at once.  The state that enters a
// segment is the sum of the end states before it, each times the decays between, the nearest first; the walk ends where the decay of
// the whole wave has gone to zero (gates of the layers, logsigmoid / 8: three segments).  Bound: the rewritten states' bytes.
// Before, up to eight segments: four elements of a state per thread, which walked the segments of their sequence and rewrote their
// chunks on the way, a memory latency each; beyond, scan and rewrite.  16 packed sequences, 32768 tokens, 4 heads of 256, with states
// 43 -> 28 us; 2 x 8192 tokens, 8 heads of 128 (16 segments each) 30.5 -> 24.5; 331 tokens, 4 heads of 128 7.3 -> 4.
// Gates that never decay read every end state before their own: as fast as the scan at 16 segments (2 x 8192 tokens, W = 64: call
// 246 -> 244 us), slower at 32 (476 -> 482; gates of the layers 478 -> 467) and at 64 (481 -> 505), so longer sequences keep the scan.
// An infinity or a NaN of an earlier segment, or of the initial state, reaches every later one whatever lies between, as it does token
// by token: where there is one (odd_words), the segments are walked in their order as the scan walks them.
// One-dimensional grid (segment slots, H, StatePart's groups), the groups fastest: there are 8, 16 or 32 of them, so the segments that
// read the same part of an end state are on one XCD.
template <int D>
__global__ __launch_bounds__(256) void state_link_kernel(const MP p) {
  __shared__ float trs[64 * 17];
  lfloat* const tr = (lfloat*)trs;
  constexpr int G = 2 * StatePart<D>::GROUPS;
  const int H = p.H, slot = blockIdx.x / (G * H), h = blockIdx.x / G % H, tid = threadIdx.x;
  int n, it0;
  segment_of(p, slot, n, it0);
  const int nchunks = p.coff[n + 1] - p.coff[n];
  if (it0 > 0 && it0 >= nchunks) return;   // (a sequence without tokens has a slot: its final state is the initial one)
  const StatePart<D> part(blockIdx.x % G, tid);
  const bool isv = part.isv;
  const int m = part.m, d = part.d;
  const int nloc = (nchunks - it0) < (1 << p.seg_sh) ? (nchunks - it0) : 1 << p.seg_sh;
  const int64_t cg0 = (int64_t)(p.coff[n] + it0) * H + h, nh = (int64_t)n * H + h;
  bf16_t* const hloc = (isv ? p.hvc : p.hkT) + (cg0 * MS + m) * D + d;
  const float* const hend = (isv ? p.hend_v : p.hend_k) + (int64_t)h * MS * D + m * D + d;   // + slot H MS D
  const float* const dtot = p.dtot + h * MS + m;                                              // + slot H MS
  Rewrite rw;
  rw.request_decays(p.dcum + cg0 * MS + m, (int64_t)H * MS, nloc);
  const bool last = it0 + nloc == nchunks;
  float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
  float own_dt = 1.f;
  if (last && p.hkt && nloc > 0) {
    own = *reinterpret_cast<const float4*>(hend + (int64_t)slot * H * MS * D);
    own_dt = dtot[(int64_t)slot * H * MS];
  }
  const int first = slot - (it0 >> p.seg_sh);
  // (the first segment itself, which has none before it, reads its own word: the walk below is the same either way)
  constexpr int Z = 2 * (D / LOCAL_DW<D>);
  const int* const words = odd_words(p) + (((int64_t)first * H + h) * Z + 2 * (d / LOCAL_DW<D>) + (isv ? 1 : 0)) * 4 + (m >> 4);
  int odd = words[(int64_t)max(min(tid & 63, slot - first - 1), 0) * H * Z * 4];
  float hs[4] = {0.f, 0.f, 0.f, 0.f}, dec = 1.f;
  for (int j = slot - 1; j >= first && __any(dec != 0.f); j -= 2) {   // the loads of two segments together
    const int j1 = j > first ? j - 1 : j;
    const float4 a = *reinterpret_cast<const float4*>(hend + (int64_t)j * H * MS * D), b = *reinterpret_cast<const float4*>(hend + (int64_t)j1 * H * MS * D);
    const float da = dtot[(int64_t)j * H * MS], db = dtot[(int64_t)j1 * H * MS];
    if (dec != 0.f) {
      hs[0] += a.x * dec; hs[1] += a.y * dec; hs[2] += a.z * dec; hs[3] += a.w * dec;
    }
    dec *= da;
    if (j > first) {
      if (dec != 0.f) {
        hs[0] += b.x * dec; hs[1] += b.y * dec; hs[2] += b.z * dec; hs[3] += b.w * dec;
      }
      dec *= db;
    }
  }
  for (int i = 64 + (tid & 63); i < slot - first; i += 64) odd |= words[(int64_t)i * H * Z * 4];
  odd = __any(odd);
  float4 h0 = make_float4(0.f, 0.f, 0.f, 0.f);
  if (p.h0k && __syncthreads_or(odd || dec != 0.f)) {
    h0 = isv ? *reinterpret_cast<const float4*>(p.h0v + (nh * MS + m) * D + d) : part.load_k(p.h0k + nh * D * MS, tr, tid);
    hs[0] += h0.x * dec; hs[1] += h0.y * dec; hs[2] += h0.z * dec; hs[3] += h0.w * dec;
  }
  if (odd) {
    hs[0] = h0.x; hs[1] = h0.y; hs[2] = h0.z; hs[3] = h0.w;
    for (int j = first; j < slot; ++j) {
      const float4 a = *reinterpret_cast<const float4*>(hend + (int64_t)j * H * MS * D);
      const float da = dtot[(int64_t)j * H * MS];
      hs[0] = hs[0] * da + a.x; hs[1] = hs[1] * da + a.y; hs[2] = hs[2] * da + a.z; hs[3] = hs[3] * da + a.w;
    }
  }
  rw.request(hloc, (int64_t)H * MS * D, fmaxf(fmaxf(fabsf(hs[0]), fabsf(hs[1])), fmaxf(fabsf(hs[2]), fabsf(hs[3]))));
  rw.store(hloc, (int64_t)H * MS * D, hs);
  if (last && p.hkt) {
    const float4 x = make_float4(hs[0] * own_dt + own.x, hs[1] * own_dt + own.y, hs[2] * own_dt + own.z, hs[3] * own_dt + own.w);
    if (isv) *reinterpret_cast<float4*>(p.hvt + (nh * MS + m) * D + d) = x;
    else part.store_k(p.hkt + nh * D * MS, x, tr, tid);
  }
}

// After state_scan_kernel: one thread per (segment, kv-head, slot, four consecutive d), every segment at once.
// grid (segment slots, H, 2*MS*D/1024): the first MS*D/4 groups of z are the k-state ([m][d]), the rest the v-state.
template <int D>
__global__ __launch_bounds__(256) void state_apply_kernel(const MP p) {
  const int H = p.H;
  const int slot = blockIdx.x, h = blockIdx.y;
  int n, it0;
  segment_of(p, slot, n, it0);
  const int nchunks = p.coff[n + 1] - p.coff[n];
  if (it0 >= nchunks) return;
  const int nloc = (nchunks - it0) < (1 << p.seg_sh) ? (nchunks - it0) : 1 << p.seg_sh;
  const int e4 = blockIdx.z * 256 + threadIdx.x;
  const bool isv = e4 >= MS * D / 4;
  const int em = (isv ? e4 - MS * D / 4 : e4) * 4;
  const int m = em / D, d = em % D;
  const int64_t sl = (int64_t)slot * H + h;
  const float4 x = *reinterpret_cast<const float4*>((isv ? p.hseg_v : p.hseg_k) + (sl * MS + m) * D + d);
  const float hs[4] = {x.x, x.y, x.z, x.w};
  const float amax = fmaxf(fmaxf(fabsf(hs[0]), fabsf(hs[1])), fmaxf(fabsf(hs[2]), fabsf(hs[3])));
  if (!(amax >= CARRY_FLOOR)) return;      // nothing is carried into this segment (its first, without initial state)
  const int64_t cg0 = (int64_t)(p.coff[n] + it0) * H + h;
  bf16_t* const hloc = (isv ? p.hvc : p.hkT) + (cg0 * MS + m) * D + d;
  Rewrite rw;
  rw.request_decays(p.dcum + cg0 * MS + m, (int64_t)H * MS, nloc);
  rw.request(hloc, (int64_t)H * MS * D, amax);
  rw.store(hloc, (int64_t)H * MS * D, hs);
}

// ==========================================================================================
// output pass
// ==========================================================================================
// One workgroup = one 64-row chunk x G query heads of one kv-head; its NW waves split the
// 64 x G query rows into RQB blocks of 16 rows per wave.  Window K/V stream through four LDS
// buffers of TK keys (two K, two V, double buffered), TK = 64 or 32 (run_mfma).
// The slot branch runs first on the same buffers: its four 64-row operand tiles (transposed
// chunk-start k-state, k_gsa rows, chunk-start v-state, v rows) fit at once when TK = 64 and
// in two stages when TK = 32.  The decay factors s_j[m] exp(gr[m] - gc_j[m]) that every wave
// needs are computed once per workgroup into LDS, already in MFMA fragment order; OWN: by the wave that uses them.

// OWN: with four waves per head every wave owns one sub-block of query rows and shares its fragments with the waves of the
// other heads at most: each forms its own in registers, and the 44 KB that hold them otherwise let a second workgroup onto
// the CU (two heads: at 128 registers, four waves per SIMD).
template <int D, int TK, bool OWN>
struct OutSmem {
  static constexpr int LDT = D + 16;
  static constexpr size_t tile_bytes = (size_t)TK * LDT * 2;
  static constexpr size_t bytes =
      4 * tile_bytes + (size_t)BT * GLD * 4 + (size_t)BT * SLD * 2 + (OWN ? 0 : (size_t)(NSEA + NSEB) * 512 * 2);
};


// SIGN: a scale that is not above zero (in the ordinary kernel the few instructions for it took 2 to 4 % of short windows: 60
// ragged documents of 300 tokens, 4 heads of 128, W = 64, 50.2 -> 52.5 us).
// EXACT: the flagged rows are formed again at the end (prefill_exact.h has when).
template <int D, int G, int NW, int TK, bool OWN, bool SIGN, bool EXACT>
__global__ __launch_bounds__(64 * NW, OWN ? NW / 2 : 1) void mfma_out_kernel(const MP p) {
  constexpr int NTHR = 64 * NW;      // threads per workgroup
  constexpr int WPU = NW / G;        // waves per (chunk, head)
  constexpr int RQB = 4 / WPU;       // 16-row query blocks per wave
  static_assert(WPU >= 1 && WPU <= 4 && RQB * WPU == 4, "bad wave split");
  static_assert(TK == 64 || TK == 32, "bad tile size");
  static_assert(!OWN || RQB == 1, "a wave's own fragments serve one sub-block");
  constexpr int KS = D / 32;
  constexpr int DB = D / 16;
  constexpr int LDT = D + 16;
  constexpr int NH = TK / 32;        // 32-key halves per tile
  constexpr int TILE = TK * LDT;
  extern __shared__ __align__(16) unsigned char smem[];
  lbf16* const tiles = (lbf16*)smem;           // K0, K1, V0, V1
  lbf16* const Kb0 = tiles;
  lbf16* const Kb1 = tiles + TILE;
  lbf16* const Vb0 = tiles + 2 * TILE;
  lbf16* const Vb1 = tiles + 3 * TILE;
  lfloat* const gcR = (lfloat*)(tiles + 4 * TILE);   // gate cumsum [row j][slot m]
  lbf16* const sR = (lbf16*)(gcR + BT * GLD);        // s [row j][slot m]
  lbf16* const SEa = sR + BT * SLD;                  // NSEA fragments of 64 lanes x 8
  lbf16* const SEb = SEa + NSEA * 512;               // NSEB fragments
  // 64-row slot-branch tiles: TK = 64 -> four buffers; TK = 32 -> two double-height buffers
  lbf16* const tA = Kb0;                                 // hkT, then (TK = 32) hv
  lbf16* const tB = TK == 64 ? Kb1 : Vb0;                // k_gsa rows, then (TK = 32) v rows
  lbf16* const tC = TK == 64 ? Vb0 : Kb0;                // hv
  lbf16* const tD = TK == 64 ? Vb1 : Vb0;                // v rows

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, kb = lane >> 4;
  const int H = p.H, HQ = p.HQ, NG = p.NG;
  // grid = (kv-head x head-group, chunk), tiles dealt so that an XCD (workgroup id % 8) streams neighbouring
  // chunks of ONE kv-head and the window tiles its resident workgroups share stay in that XCD's L2 (xcd_tile;
  // with 8 (kv-head, group) pairs that is the launch order itself).  Chunks are taken from
  // the last to the first: the chunks at the start of a sequence have the shortest windows, and
  // short workgroups at the end of the launch leave the smallest tail.
  const int ngrp = NG / G;
  int vx, vy;
  xcd_tile(ngrp, p.NT, vx, vy);
  const int chunk = p.NT - 1 - vy;
  const int h = vx / ngrp, grp = vx % ngrp;
  const int hq = h * NG + grp * G + wave / WPU;
  const int qb0 = (wave % WPU) * RQB;
  const int n = p.cidx[2 * chunk], it = p.cidx[2 * chunk + 1];
  const int bos = p.cu[n], eos = p.cu[n + 1];
  const int c0 = bos + it * BT;
  const int rows = (eos - c0) < BT ? (eos - c0) : BT;
  // logits are kept unscaled; p = exp2(cs * (s - m)) with cs > 0: the sign of the scale is the queries', and where it is 0 they are
  const float cs = !SIGN ? p.scale * LOG2E : p.scale == 0.f ? LOG2E : fabsf(p.scale) * LOG2E;
  auto query = [&](const uint4& x) {
    if constexpr (!SIGN) return as_bf16x8(x);
    const uint32_t keep = p.scale == 0.f ? 0u : ~0u, sign = p.scale < 0.f ? 0x80008000u : 0u;
    return as_bf16x8(make_uint4((x.x & keep) ^ sign, (x.y & keep) ^ sign, (x.z & keep) ^ sign, (x.w & keep) ^ sign));
  };
  const int64_t cg = (int64_t)chunk * H + h;
  int exact = 0;   // 16-row blocks of the chunk that decay too fast for the split decay (flags of the state pass)
  if constexpr (EXACT) exact = p.flags[cg * 4] | p.flags[cg * 4 + 1] | p.flags[cg * 4 + 2] | p.flags[cg * 4 + 3];

  // ---- window tile schedule: tile i covers keys [c0 + 64 - TK (i+1), c0 + 64 - TK i) ----------
  int lowest = bos;
  if (p.wl >= 0 && c0 - p.wl > bos) lowest = c0 - p.wl;
  const int ntiles = (c0 + 64 - lowest + TK - 1) / TK;
  TileRegs<TK, D, NTHR> rk, rv;
  // Tile boundaries are multiples of TK away from bos, so a window tile never starts before its
  // sequence; only the tiles over the chunk's own rows can run past eos.  Every tile that ends at
  // or before eos is loaded unconditionally from a wave-uniform base plus per-thread 32-bit
  // offsets that never change (one scalar subtraction per tile instead of per-load 64-bit
  // address arithmetic); the others take the row-checked path.
  constexpr int NPC = TK * D / 8 / NTHR;   // 16-byte pieces per thread and tile
  uint32_t goff[NPC], loff[NPC];
#pragma unroll
  for (int u = 0; u < NPC; ++u) {
    const int c = tid + NTHR * u;
    const int row = c / (D / 8), col = (c % (D / 8)) * 8;
    goff[u] = (uint32_t)row * (uint32_t)(H * D) + col;
    loff[u] = row * (D + 16) + col;
  }
  auto issue_window_fast = [&](int i) {
    const int64_t grow0 = (int64_t)c0 + 64 - TK * (i + 1);
    const bf16_t* kb_ = p.k_swa + (grow0 * H + h) * D;
    const bf16_t* vb_ = p.v + (grow0 * H + h) * D;
#pragma unroll
    for (int u = 0; u < NPC; ++u) {
      rk.r[u] = *reinterpret_cast<const uint4*>(kb_ + goff[u]);
      rv.r[u] = *reinterpret_cast<const uint4*>(vb_ + goff[u]);
    }
  };
  // tiles 0 and 1 (issued before the loop) may cover rows of the chunk itself, i.e. run past eos
  auto issue_window = [&](int i) {
    const int64_t grow0 = (int64_t)c0 + 64 - TK * (i + 1);
    if (grow0 + TK > eos) {
      int vhi = eos - (int)grow0;
      vhi = vhi < 0 ? 0 : (vhi > TK ? TK : vhi);
      tile_g2r<TK, D, NTHR>(rk, p.k_swa + (int64_t)h * D, (int64_t)H * D, grow0, 0, vhi, tid);
      tile_g2r<TK, D, NTHR>(rv, p.v + (int64_t)h * D, (int64_t)H * D, grow0, 0, vhi, tid);
    } else {
      issue_window_fast(i);
    }
  };
  auto stage_window = [&](lbf16* kdst, lbf16* vdst) {
#pragma unroll
    for (int u = 0; u < NPC; ++u) {
      lds_st16(kdst + loff[u], rk.r[u]);
      lds_st16(vdst + loff[u], rv.r[u]);
    }
  };
  // ---- phase 0: slot-branch operands -> LDS --------------------------------------------------
  int vlo = p.shift - it * BT;
  vlo = vlo < 0 ? 0 : vlo;
  const int64_t grow_s = (int64_t)c0 - p.shift;
  // Every global load of this phase is issued before the first result is used, so the phase costs
  // one memory latency, not one per tile.
  // chunk-start states are plain [m][d] bf16 tiles (the state pass leaves the true states)
  auto issue_state = [&](TileRegs<BT, D, NTHR>& r, const bf16_t* hst) {
    tile_g2r<BT, D, NTHR>(r, hst + cg * MS * D, (int64_t)D, 0, 0, BT, tid);
  };
  auto load_state_tile = [&](lbf16* dst, const bf16_t* hst) {
    TileRegs<BT, D, NTHR> r;
    issue_state(r, hst);
    tile_r2l<BT, D, NTHR>(dst, r, tid);
  };
  auto load_rows_tile = [&](lbf16* dst, const bf16_t* src) {
    TileRegs<BT, D, NTHR> t;
    tile_g2r<BT, D, NTHR>(t, src + (int64_t)h * D, (int64_t)H * D, grow_s, vlo, rows, tid);
    tile_r2l<BT, D, NTHR>(dst, t, tid);
  };
  {
    TileRegs<BT, D, NTHR> ra, rc, tb, td;
    constexpr int NG4 = 1024 / NTHR, NS8 = (512 + NTHR - 1) / NTHR;
    float4 gx[NG4];
    uint4 sx[NS8];
    issue_state(ra, p.hkT);
    tile_g2r<BT, D, NTHR>(tb, p.k_gsa + (int64_t)h * D, (int64_t)H * D, grow_s, vlo, rows, tid);
    if (TK == 64) {
      issue_state(rc, p.hvc);
      tile_g2r<BT, D, NTHR>(td, p.v + (int64_t)h * D, (int64_t)H * D, grow_s, vlo, rows, tid);
    }
    // gate cumsum table (fp32 [64][64]); rows past the sequence end are zero
    const float* gsrc = p.gc + cg * BT * MS;
#pragma unroll
    for (int u = 0; u < NG4; ++u) {
      const int c4 = tid + NTHR * u;
      const int j = c4 >> 4, m4 = (c4 & 15) * 4;
      gx[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (j < rows) gx[u] = *reinterpret_cast<const float4*>(gsrc + j * MS + m4);
    }
    // s rows of the slot branch (shifted)
#pragma unroll
    for (int u = 0; u < NS8; ++u) {
      const int c8 = tid + NTHR * u;
      const int j = c8 >> 3, m8 = (c8 & 7) * 8;
      sx[u] = make_uint4(0, 0, 0, 0);
      if (c8 < 512 && j >= vlo && j < rows) sx[u] = *reinterpret_cast<const uint4*>(p.s + ((grow_s + j) * H + h) * MS + m8);
    }
    issue_window(0);
    __builtin_amdgcn_sched_barrier(0);
    tile_r2l<BT, D, NTHR>(tA, ra, tid);
    tile_r2l<BT, D, NTHR>(tB, tb, tid);
    if (TK == 64) {
      tile_r2l<BT, D, NTHR>(tC, rc, tid);
      tile_r2l<BT, D, NTHR>(tD, td, tid);
    }
#pragma unroll
    for (int u = 0; u < NG4; ++u) {
      const int c4 = tid + NTHR * u;
      const int j = c4 >> 4, m4 = (c4 & 15) * 4;
      *reinterpret_cast<NHA_LDS f32x4*>(gcR + j * GLD + m4) = (f32x4){gx[u].x, gx[u].y, gx[u].z, gx[u].w};
    }
#pragma unroll
    for (int u = 0; u < NS8; ++u) {
      const int c8 = tid + NTHR * u;
      const int j = c8 >> 3, m8 = (c8 & 7) * 8;
      if (c8 < 512) lds_st16(sR + j * SLD + m8, sx[u]);
    }
  }
  __syncthreads();
  // decay-factor fragments, one (fragment, lane) item = 8 values.  Sub-block Q (16 query rows)
  // references the gate cumsum gr of the row before it: exponent gr[m] - gc_j[m] <= 0 for rows
  // j of earlier sub-blocks, and bounded by the sub-block's own decay for its diagonal rows.
  // All LDS reads of an item are issued before the first exponential waits for one: read one at a
  // time, the 8 values of an item cost 24 LDS latencies in sequence.
  // sea_item: s_j[m] exp(gr[m] - gc_j[m]) with a slot per lane (rows j of blocks 2 pr and 2 pr + 1, slots of block mb)
  auto sea_item = [&](int Q, int pr, int mb, int fl16, int fkb) {
    const int m = 16 * mb + fl16;
    const float gr = Q > 0 ? gcR[(16 * Q - 1) * GLD + m] : 0.f;
    float gv[8];
    bf16_t sv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int j = 16 * (2 * pr + (e >> 2)) + 4 * fkb + (e & 3);   // j < 64 for every fragment
      gv[e] = gcR[j * GLD + m];
      sv[e] = sR[j * SLD + m];
    }
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int jb = 2 * pr + (e >> 2);
      const float val = bf16_to_f32(sv[e]) * fexp(fminf(gr - gv[e], DECAY_CLAMP));
      out[e] = (__bf16)(jb <= Q ? val : 0.f);
    }
    return out;
  };
  // seb_item: the same with a row j of block jb per lane (slots of half pr)
  auto seb_item = [&](int Q, int jb, int pr, int fl16, int fkb) {
    const int j = 16 * jb + fl16;
    f32x4 gv[2], gr[2];
    bf16x4 sv[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int m0 = 32 * pr + 16 * hh + 4 * fkb;   // the lane's 4 consecutive slots of this half
      gv[hh] = *reinterpret_cast<const NHA_LDS f32x4*>(gcR + j * GLD + m0);
      gr[hh] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (Q > 0) gr[hh] = *reinterpret_cast<const NHA_LDS f32x4*>(gcR + (16 * Q - 1) * GLD + m0);
      sv[hh] = *reinterpret_cast<const NHA_LDS bf16x4*>(sR + j * SLD + m0);
    }
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      out[e] = (__bf16)((float)sv[e >> 2][e & 3] * fexp(fminf(gr[e >> 2][e & 3] - gv[e >> 2][e & 3], DECAY_CLAMP)));
    return out;
  };
  if constexpr (!OWN) {
    for (int item = tid; item < (NSEA + NSEB) * 64; item += NTHR) {
      const int f = item >> 6, ln = item & 63;
      if (f < NSEA) {
        const int Q = f < 4 ? 0 : f < 8 ? 1 : f < 16 ? 2 : 3;
        const int rem = f - sea_base(Q);
        *reinterpret_cast<NHA_LDS bf16x8*>(SEa + f * 512 + ln * 8) = sea_item(Q, rem >> 2, rem & 3, ln & 15, ln >> 4);
      } else {
        const int g2 = f - NSEA;
        const int Q = g2 < 2 ? 0 : g2 < 6 ? 1 : g2 < 12 ? 2 : 3;
        const int rem = g2 - seb_base(Q);
        *reinterpret_cast<NHA_LDS bf16x8*>(SEb + g2 * 512 + ln * 8) = seb_item(Q, rem >> 1, rem & 1, ln & 15, ln >> 4);
      }
    }
    __syncthreads();
  }

  // per-lane softmax state for the RQB queries (l16 + 16*(qb0+qb)) this lane serves
  float mrun[RQB], lg[RQB];
  f32x4 O[DB][RQB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int qb = 0; qb < RQB; ++qb) O[db][qb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  bf16x8 bp[RQB][2], bpr[RQB][2];   // slot probabilities x exp(gc_i) and x exp(gc_i - gr), B operands

  // window-query fragments: requested here so that they land during the slot branch
  bf16x8 qs[RQB][KS];
#pragma unroll
  for (int qb = 0; qb < RQB; ++qb) {
    const int irow = 16 * (qb0 + qb) + l16;
    const bf16_t* qp = p.q_swa + ((int64_t)(c0 + irow) * HQ + hq) * D + 8 * kb;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 x = make_uint4(0, 0, 0, 0);
      if (irow < rows) x = *reinterpret_cast<const uint4*>(qp + 32 * ks);
      qs[qb][ks] = query(x);
    }
  }
  // ---- phase 1a: slot logits and the slot "tile" of the softmax, one 16-row block at a time ----
#pragma unroll
  for (int qb = 0; qb < RQB; ++qb) {
    const int Q = qb0 + qb;                // sub-block index inside the chunk
    const int irow = 16 * Q + l16;         // this lane's query row inside the chunk
    bf16x8 qf[KS];
    {
      const bf16_t* qp = p.q_gsa + ((int64_t)(c0 + irow) * HQ + hq) * D + 8 * kb;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        uint4 x = make_uint4(0, 0, 0, 0);
        if (irow < rows) x = *reinterpret_cast<const uint4*>(qp + 32 * ks);
        qf[ks] = query(x);
      }
    }
    // inter-chunk slot logits: okT[m][i] = sum_d hkT[m][d] q[i][d]
    f32x4 ok[4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) ok[mb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) ok[mb] = mfma16(lds_frag(tA, LDT, 16 * mb + l16, 32 * ks + 8 * kb), qf[ks], ok[mb]);
    // intra-chunk scores AT[j][i] = sum_d k_gsa[j][d] q[i][d] for row blocks jb <= Q, masked j <= i
    bf16x8 bA[2];
    {
      f32x4 at[4];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) at[jb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int jb = 0; jb < 4; ++jb)
          if (jb <= Q) at[jb] = mfma16(lds_frag(tB, LDT, 16 * jb + l16, 32 * ks + 8 * kb), qf[ks], at[jb]);
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
    // okT_intra[m][i] = sum_j s_j[m] exp(gr[m] - gc_j[m]) AT[j][i]
    f32x4 oki[4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      oki[mb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int pr = 0; pr < 2; ++pr)
        if (2 * pr <= Q) {
          bf16x8 se;
          if constexpr (OWN) se = sea_item(Q, pr, mb, l16, kb);
          else se = *reinterpret_cast<const NHA_LDS bf16x8*>(SEa + (sea_base(Q) + 4 * pr + mb) * 512 + lane * 8);
          oki[mb] = mfma16(se, bA[pr], oki[mb]);
        }
    }
    // combine, then the slot "tile" of the online softmax (logits unscaled, exponent scale cs)
    const int rref = 16 * Q - 1;
    float rmax = -INFINITY;
    f32x4 egi[4], egr[4];   // exp(gc_i[m]) and exp(gc_i[m] - gr[m]) in accumulator layout
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const float4 gi = lds_ld_f4(gcR + irow * GLD + 16 * mb + 4 * kb);
      float4 gr4 = make_float4(0.f, 0.f, 0.f, 0.f);
      if (Q > 0) gr4 = lds_ld_f4(gcR + rref * GLD + 16 * mb + 4 * kb);
      const float giv[4] = {gi.x, gi.y, gi.z, gi.w};
      const float grv[4] = {gr4.x, gr4.y, gr4.z, gr4.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        egi[mb][r] = fexp(giv[r]);
        egr[mb][r] = fexp(giv[r] - grv[r]);
        ok[mb][r] = ok[mb][r] * egi[mb][r] + oki[mb][r] * egr[mb][r];
        rmax = fmaxf(rmax, ok[mb][r]);
      }
    }
    rmax = max_over_rows(rmax);
    mrun[qb] = rmax;
    float psum = 0.f;
    const float mc = rmax * cs;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ok[mb][r] = fexp2(ok[mb][r] * cs - mc);   // unnormalised slot probabilities
        psum += ok[mb][r];
      }
    lg[qb] = psum;   // partial over this lane's 16 slots
    if (p.lse_gsa) {
      float tot = psum + __shfl_xor(psum, 16, 64);
      tot += __shfl_xor(tot, 32, 64);
      if (kb == 0 && irow < rows) p.lse_gsa[(int64_t)(c0 + irow) * HQ + hq] = (mc + __builtin_amdgcn_logf(tot)) * LN2;
    }
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
      bp[qb][pr] = pack8(x0, x1);
      bpr[qb][pr] = pack8(y0, y1);
    }
  }
  if (TK == 32) {
    // second stage of the slot-branch tiles: the state / row tiles of the value side
    __syncthreads();
    load_state_tile(tC, p.hvc);
    load_rows_tile(tD, p.v);
    __syncthreads();
  }
  // ---- phase 1b: slot read ----------------------------------------------------------------------
#pragma unroll
  for (int qb = 0; qb < RQB; ++qb) {
    const int Q = qb0 + qb;
    // inter-chunk part: O^T[d][i] += sum_m hv[m][d] (p[i][m] exp(gc_i[m]))
#pragma unroll
    for (int pr = 0; pr < 2; ++pr)
#pragma unroll
      for (int db = 0; db < DB; ++db)
        O[db][qb] = mfma16(lds_frag_tr(tC, LDT, 32 * pr, 32 * pr + 16, 16 * db, lane), bp[qb][pr], O[db][qb]);
    // intra-chunk part: AvT[j][i] = sum_m s_j[m] exp(gr[m]-gc_j[m]) (p[i][m] exp(gc_i[m]-gr[m])), j <= i
    bf16x8 bAv[2];
    {
      f32x4 av[4];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        av[jb] = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (jb <= Q) {
#pragma unroll
          for (int pr = 0; pr < 2; ++pr) {
            bf16x8 se;
            if constexpr (OWN) se = seb_item(Q, jb, pr, l16, kb);
            else se = *reinterpret_cast<const NHA_LDS bf16x8*>(SEb + (seb_base(Q) + 2 * jb + pr) * 512 + lane * 8);
            av[jb] = mfma16(se, bpr[qb][pr], av[jb]);
          }
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
#pragma unroll
    for (int pr = 0; pr < 2; ++pr)
      if (2 * pr <= Q) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
          O[db][qb] = mfma16(lds_frag_tr(tD, LDT, 32 * pr, 32 * pr + 16, 16 * db, lane), bAv[pr], O[db][qb]);
      }
  }
  // ---- phase 2: sliding window, streamed in TK-key tiles --------------------------------------
  lds_barrier();   // every wave is done with the slot-branch tiles
  stage_window(Kb0, Vb0);
  if (ntiles > 1) issue_window(1);
  lds_barrier();

  // lazy rescaling: the running reference max only moves when a half tile exceeds it by more than
  // 2^RESCALE_LOG2 in probability units, so O is rescaled a handful of times per chunk
  constexpr float RESCALE_LOG2 = 8.f;
  const float thr = RESCALE_LOG2 / cs;
  f32x4 Lw[RQB];
#pragma unroll
  for (int qb = 0; qb < RQB; ++qb) Lw[qb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;
  // every load issued before the prefetch of tile 1 (queries, tile 0) has landed here, so inside
  // the loop only the tile prefetch of the previous iteration is ever outstanding
  __builtin_amdgcn_s_waitcnt(0x0f70 | (2 * NPC));   // vmcnt(2 * NPC), other counters untouched
  for (int i = 0; i < ntiles; ++i) {
    const int cur = i & 1;
    const lbf16* Kt = cur ? Kb1 : Kb0;
    const lbf16* Vt = cur ? Vb1 : Vb0;
    const int xbase = 64 - TK * (i + 1);   // key offset of the tile's first key relative to the chunk start
    const bool edge = (xbase + TK - 1 > 0) || (p.wl >= 0 && p.wl < TK * (i + 1) - 1);
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) {
      // S^T[key][q] for the 32 keys of this half: 2 key blocks x RQB query blocks, the
      // 2 * RQB accumulators advance together so consecutive MFMAs are independent
      f32x4 S[2][RQB];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int qb = 0; qb < RQB; ++qb) S[kk][qb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bf16x8 a0 = lds_frag(Kt, LDT, 32 * hf + l16, 32 * ks + 8 * kb);
        const bf16x8 a1 = lds_frag(Kt, LDT, 32 * hf + 16 + l16, 32 * ks + 8 * kb);
#pragma unroll
        for (int qb = 0; qb < RQB; ++qb) {
          S[0][qb] = mfma16(a0, qs[qb][ks], S[0][qb]);
          S[1][qb] = mfma16(a1, qs[qb][ks], S[1][qb]);
        }
      }
      if (edge) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int qb = 0; qb < RQB; ++qb) {
            const int y = 16 * (qb0 + qb) + l16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int x = xbase + 32 * hf + 16 * kk + 4 * kb + r;
              const bool ok = (x <= y) && (p.wl < 0 || x >= y - p.wl);
              if (!ok) S[kk][qb][r] = -INFINITY;
            }
          }
      }
      // online softmax per query column
      bf16x8 P[RQB];
      bool need = false;
      float rmax[RQB];
#pragma unroll
      for (int qb = 0; qb < RQB; ++qb) {
        float x = fmaxf(fmaxf(S[0][qb][0], S[0][qb][1]), fmaxf(S[0][qb][2], S[0][qb][3]));
        x = fmaxf(x, fmaxf(fmaxf(S[1][qb][0], S[1][qb][1]), fmaxf(S[1][qb][2], S[1][qb][3])));
        // the lane's own 8 keys suffice to decide (some lane exceeds the threshold iff the column
        // maximum does); the cross-lane maximum is only formed on the rare rescale path
        rmax[qb] = x;
        need |= x > mrun[qb] + thr;
      }
      if (__any(need)) {
#pragma unroll
        for (int qb = 0; qb < RQB; ++qb) {
          const float mnew = fmaxf(mrun[qb], max_over_rows(rmax[qb]));
          const float alpha = fexp2((mrun[qb] - mnew) * cs);
          mrun[qb] = mnew;
          lg[qb] *= alpha;
#pragma unroll
          for (int r = 0; r < 4; ++r) Lw[qb][r] *= alpha;
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int r = 0; r < 4; ++r) O[db][qb][r] *= alpha;
        }
      }
#pragma unroll
      for (int qb = 0; qb < RQB; ++qb) {
        const float mc = mrun[qb] * cs;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[kk][qb][r] = fexp2(S[kk][qb][r] * cs - mc);
        P[qb] = pack8(S[0][qb], S[1][qb]);
        // window row sums on the matrix core: every row of ones^T P is the sum over the 32 keys
        Lw[qb] = mfma16(ones, P[qb], Lw[qb]);
      }
      // O^T[d][q] += V^T P^T over the 32 keys of this half
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const bf16x8 a = lds_frag_tr(Vt, LDT, 32 * hf, 32 * hf + 16, 16 * db, lane);
#pragma unroll
        for (int qb = 0; qb < RQB; ++qb) O[db][qb] = mfma16(a, P[qb], O[db][qb]);
      }
    }
    if (i + 1 < ntiles) {
      stage_window(cur ? Kb0 : Kb1, cur ? Vb0 : Vb1);
      if (i + 2 < ntiles) issue_window_fast(i + 2);   // tiles >= 2 lie wholly before the chunk
    }
    lds_barrier();
  }

  // ---- epilogue -------------------------------------------------------------------------------
#pragma unroll
  for (int qb = 0; qb < RQB; ++qb) {
    const int irow = 16 * (qb0 + qb) + l16;
    const float lwt = Lw[qb][0];
    float lgt = lg[qb] + __shfl_xor(lg[qb], 16, 64);
    lgt += __shfl_xor(lgt, 32, 64);
    const float inv = 1.f / (lwt + lgt);
    if (irow < rows) {
      bf16_t* op = p.o + ((int64_t)(c0 + irow) * HQ + hq) * D + 4 * kb;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        bf16x4 pk;
#pragma unroll
        for (int r = 0; r < 4; ++r) pk[r] = (__bf16)(O[db][qb][r] * inv);
        *reinterpret_cast<bf16x4*>(op + 16 * db) = pk;
      }
      if (p.lse_swa && kb == 0)
        p.lse_swa[(int64_t)(c0 + irow) * HQ + hq] = (mrun[qb] * cs + __builtin_amdgcn_logf(lwt)) * LN2;
    }
  }
  if constexpr (EXACT) {
    if (exact == 0) return;
    before_exact();
    exact_rows<D, NTHR / 256, false>(arguments_again(), reinterpret_cast<float*>(smem), chunk, h, h * NG + grp * G, G, exact);
  }
}

// ==========================================================================================
// exact recomputation of the flagged rows (prefill_exact.h) after the output passes that do not do it themselves: grid (chunk, kv-head),
// the q-heads of the group in turn; workgroups of unflagged chunks leave at once
// ==========================================================================================
template <int D>
__global__ __launch_bounds__(256) void mfma_repair_kernel(const MP p) {
  const int chunk = blockIdx.x, h = blockIdx.y;
  const int* fl = p.flags + ((int64_t)chunk * p.H + h) * 4;
  const int bits = fl[0] | fl[1] | fl[2] | fl[3];
  if (bits == 0) return;
  extern __shared__ __align__(16) float rsm[];
  exact_rows<D, 1>(p, rsm, chunk, h, h * p.NG, p.NG, bits);
}

template <int D>
int launch_repair(const MP& p, hipStream_t st) {
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  const size_t lds = ExactSmem<D, 1, true>::bytes;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute((const void*)mfma_repair_kernel<D>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
  if (attr_err != hipSuccess) {
    set_error("nha_prefill_fwd(mfma): cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(attr_err));
    return NHA_ERR_LAUNCH;
  }
  hipLaunchKernelGGL((mfma_repair_kernel<D>), dim3(p.NT, p.H), dim3(256), lds, st, p);
  NHA_CHECK_LAUNCH("nha_prefill_fwd(mfma repair pass)");
  return NHA_OK;
}

template <int D, int G, int NW, int TK, bool OWN, bool SIGN, bool EXACT>
int launch_out_of(const MP& p, hipStream_t st) {
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  constexpr size_t own = OutSmem<D, TK, OWN>::bytes, rows = EXACT ? ExactSmem<D, NW / 4, false>::bytes : 0;
  constexpr size_t lds = own > rows ? own : rows;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute((const void*)mfma_out_kernel<D, G, NW, TK, OWN, SIGN, EXACT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
  if (attr_err != hipSuccess) {
    set_error("nha_prefill_fwd(mfma): cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(attr_err));
    return NHA_ERR_LAUNCH;
  }
  hipLaunchKernelGGL((mfma_out_kernel<D, G, NW, TK, OWN, SIGN, EXACT>), dim3(p.H * (p.NG / G), p.NT), dim3(64 * NW), lds, st, p);
  NHA_CHECK_LAUNCH("nha_prefill_fwd(mfma output pass)");
  return NHA_OK;
}
template <int D, int G, int NW, int TK, bool OWN>
int launch_out(const MP& p, bool* exact, hipStream_t st) {
  if (!(p.scale > 0.f)) return launch_out_of<D, G, NW, TK, OWN, true, false>(p, st);
  // One or two heads at head sizes 64 and 128 (not the eight waves of two heads that have their own fragments and 128 registers: the
  // code for the rows spills 50 of them); at D = 64, where the pass is short: a workgroup takes 14 us and 0.6 per unit.
  if constexpr (D <= 128 && (G == 1 || (G == 2 && !OWN))) {
    constexpr int PER_CU = !OWN ? 1 : D == 64 ? 3 : 2;
    *exact = D == 128 || (double)p.NT * p.HQ / G / (256 * PER_CU) * (14 + 0.6 * window_units(p)) <= EXACT_INSIDE_US;
    if (*exact) return launch_out_of<D, G, NW, TK, OWN, false, true>(p, st);
  }
  return launch_out_of<D, G, NW, TK, OWN, false, false>(p, st);
}

// state pass: level 1, then level 2 in the forward form (true chunk-start states in place) or, for
// the backward's state export, in the segment form (segment-start states beside the local ones)
template <int D>
int run_state_pass(const MP& p, bool segment_form, hipStream_t st) {
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  constexpr int DW = LOCAL_DW<D>;
  const size_t lds = (size_t)BT * (DW + 16) * 2 + (size_t)2 * BT * SLD * 2;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute((const void*)mfma_state_local_kernel<D, DW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
  if (attr_err != hipSuccess) {
    set_error("nha_prefill_fwd(mfma): cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(attr_err));
    return NHA_ERR_LAUNCH;
  }
  // at most NT / segment + N segments: every sequence but for its last segment fills them
  const int nslot = (p.NT >> p.seg_sh) + p.N;
  const int64_t l1_grid = (int64_t)nslot * p.H * 2 * (D / DW);
  if (l1_grid > 0x7fffffff) {
    set_error("nha_prefill_fwd(mfma): too many segments for one launch (%lld workgroups)", (long long)l1_grid);
    return NHA_ERR_UNSUPPORTED;
  }
  hipLaunchKernelGGL((mfma_state_local_kernel<D, DW>), dim3((unsigned)l1_grid), dim3(256), lds, st, p);
  NHA_CHECK_LAUNCH("nha_prefill_fwd(mfma state pass, level 1)");
  const int64_t link_grid = segment_form ? 0 : state_link_grid(p.NT, p.N, p.H, D, p.seg_sh);
  if (link_grid) {
    hipLaunchKernelGGL((state_link_kernel<D>), dim3((unsigned)link_grid), dim3(256), 0, st, p);
  } else {
    hipLaunchKernelGGL((state_scan_kernel<D>), dim3(p.N * p.H, 2 * MS * D / 1024), dim3(256), 0, st, p);
    if (!segment_form) hipLaunchKernelGGL((state_apply_kernel<D>), dim3(nslot + 1, p.H, 2 * MS * D / 1024), dim3(256), 0, st, p);
  }
  NHA_CHECK_LAUNCH("nha_prefill_fwd(mfma state pass, level 2)");
  return NHA_OK;
}

template <int D>
int run_mfma(const MP& p, int phases, hipStream_t st) {
  if (p.NT > 65535) {
    set_error("nha_prefill_fwd(mfma): more than 65535 chunks (%d) in one call", p.NT);
    return NHA_ERR_UNSUPPORTED;
  }
  if (phases != 2) {
    const int rc = run_state_pass<D>(p, false, st);
    if (rc != NHA_OK) return rc;
  }
  if (phases != 1) {
    // G query heads of one kv-head share a workgroup.  D <= 128: 64-key tiles, 8 waves of 32 (G = 4)
    // or 16 (G = 2) query rows, two per SIMD; D = 256: 32-key tiles and 16-row waves to fit the
    // register file and LDS.  One head (G = 1): 32-key tiles, four waves and two (D = 128) or three
    // (D = 64) workgroups per CU, which 64-key tiles or decay fragments in LDS do not leave room for:
    // 16 heads, 8192 tokens, W = 2048: D = 64 291 -> 147 us, D = 128 434 -> 269 us (with 64-key tiles 165, 375);
    // 5003 packed tokens, W = 300: 93 -> 46, 119 -> 70.  G = 2: where there is more than a workgroup for
    // every CU, two fit one as well (8 / 4 heads, 4 x 8000 tokens, W = 1500: D = 128 378 -> 330-353 us, with 32-key tiles; D = 64
    // 244 -> 198); below, one with the fragments shared is faster (3000 tokens, 188 workgroups: 25 against 31, 17.5 against 19)
    int rc;
    bool exact = false;   // the output pass has formed the flagged rows itself
#ifdef NHA_AB_SWITCHES   // measurement builds only (-DNHA_AB_SWITCHES): run the kernels the LDS-direct ones replaced
    static const bool ring_off = getenv("NHA_PREFILL_NO_RING") != nullptr;
#else
    constexpr bool ring_off = false;
#endif
    if (!ring_off && prefill_ring_supported(p, D)) return prefill_ring_launch(p, D, st);
    if (!ring_off && prefill_ring256_supported(p, D)) return prefill_ring256_launch(p, st);
    if constexpr (D <= 128) {
      if (p.NG % 4 == 0) rc = launch_out<D, 4, 8, 64, false>(p, &exact, st);
      else if (p.NG % 2 == 0 && (int64_t)p.HQ / 2 * p.NT > 256) rc = launch_out<D, 2, 8, D == 128 ? 32 : 64, true>(p, &exact, st);
      else if (p.NG % 2 == 0) rc = launch_out<D, 2, 8, 64, false>(p, &exact, st);
      else rc = launch_out<D, 1, 4, 32, true>(p, &exact, st);
    } else {
      if (p.NG % 2 == 0) rc = launch_out<D, 2, 8, 32, false>(p, &exact, st);
      else rc = launch_out<D, 1, 4, 32, true>(p, &exact, st);
    }
    return rc != NHA_OK || exact ? rc : launch_repair<D>(p, st);
  }
  return NHA_OK;
}

static size_t aligned(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace

// A launch holds fewer than 2^32 threads, 2^24 workgroups here; scan and rewrite, whose grids have three dimensions, take larger calls
// (65535 sequences of one chunk, 16 kv-heads of 128: 33 M).
int64_t state_link_grid(int NT, int N, int H, int D, int seg_sh) {
  const int64_t grid = ((int64_t)(NT >> seg_sh) + N) * H * (2 * MS * D / 1024);
  return (int64_t)NT <= ((int64_t)LINK_SEGS * N << seg_sh) && grid < 1 << 24 ? grid : 0;
}

bool prefill_mfma_supported(const NhaPrefillArgs* a) {
  return a->dtype == NHA_DTYPE_BF16 && a->K == a->V && (a->K == 64 || a->K == 128 || a->K == 256) && a->M == MS;
}

namespace {
struct ScratchPlan {
  size_t hkT, hvc, gc, dcum, hend_k, hend_v, hseg_k, hseg_v, dtot, flags, total;
  int seg_sh;
};
ScratchPlan plan_scratch(const NhaPrefillArgs* a, int seg_sh) {
  const size_t per = (size_t)a->NT * a->H;
  const size_t nslot = ((size_t)a->NT >> seg_sh) + a->N + 1;
  const size_t seg = aligned(nslot * a->H * MS * a->K * 4);
  ScratchPlan s;
  size_t off = 0;
  s.hkT = off; off += aligned(per * MS * a->K * 2);
  s.hvc = off; off += aligned(per * MS * a->V * 2);
  s.gc = off; off += aligned(per * BT * MS * 4);
  s.dcum = off; off += aligned(per * MS * 4);
  s.hend_k = off; off += seg;
  s.hend_v = off; off += seg;
  s.hseg_k = off; off += seg;
  s.hseg_v = off; off += seg;
  s.dtot = off; off += aligned(nslot * a->H * MS * 4);
  s.flags = off; off += aligned(per * 4 * 4);
  s.total = off;
  s.seg_sh = seg_sh;
  return s;
}

// Chunks per segment: 8, where the chip is full.  Level 1 walks its segment at 2 us per chunk whatever else runs, so a call that leaves
// places on the chip empty takes shorter segments, as long as all its workgroups are resident at once (two per CU at head sizes 128 and
// 256, three at 64, by registers); level 2 then combines more of them.  The weights 11 : 1 are those of level 2 as a chain over the segments,
// about 0.25 us each, as in the backward and in sequences of more than LINK_SEGS segments; in one launch a segment costs 0.3 us with
// slow gates and 0.2 with fast ones.  Level 1 + level 2 in one launch, slow gates, with 8, 4, 2 and 1 chunks, us: 1000 tokens, 8 kv-heads of
// 128 24.2 + 5.0, 16.3 + 5.5, 12.9 + 6.5, 11.9 + 9.7; 4 of 256 23.4 + 4.9, 16.2 + 5.0, 13.4 + 6.0, 12.5 + 9.4; so there the rule takes 1 chunk
// where 2 would be 1 to 2 us faster.  More workgroups than places lose: 2 x 2048 tokens, 8 heads of 128 32.5 us with 8 chunks, 26.0 with
// 4, 29.1 with 2.
// A call whose workspace fits the library's own array with 8 chunks keeps fitting it.
ScratchPlan plan_scratch(const NhaPrefillArgs* a) {
  const ScratchPlan full = plan_scratch(a, 3);
  const int z = a->K >= 256 ? 4 : 2, places = a->K >= 128 ? 512 : 768;
  const int64_t chunks = ((int64_t)a->NT + a->N - 1) / a->N;
  int best = 3;
  for (int sh = 2; sh >= 0; --sh) {
    if ((((int64_t)a->NT >> sh) + a->N) * a->H * z > places) break;
    if ((11 << sh) + (chunks >> sh) >= (11 << best) + (chunks >> best)) break;
    if (full.total <= (size_t)NHA_NOALLOC_SCRATCH_BYTES && plan_scratch(a, sh).total > (size_t)NHA_NOALLOC_SCRATCH_BYTES) break;
    best = sh;
  }
  return best == 3 ? full : plan_scratch(a, best);
}

// The plan of a call: the best one that a->scratch_bytes holds.  Short segments take up to three times the room, so a workspace
// that was sized for a longer call may be too small for a shorter one's best plan; eight chunks fit it always.
ScratchPlan plan_call(const NhaPrefillArgs* a) {
  ScratchPlan s = plan_scratch(a);
  while (s.seg_sh < 3 && s.total > a->scratch_bytes) s = plan_scratch(a, s.seg_sh + 1);
  return s;
}
}  // namespace

size_t prefill_mfma_scratch_bytes(const NhaPrefillArgs* a) { return plan_scratch(a).total; }
size_t prefill_mfma_least_scratch_bytes(const NhaPrefillArgs* a) { return plan_scratch(a, 3).total; }

namespace {
MP make_mp(const NhaPrefillArgs* a) {
  MP p;
  p.q_swa = (const bf16_t*)a->q_swa; p.k_swa = (const bf16_t*)a->k_swa;
  p.q_gsa = (const bf16_t*)a->q_gsa; p.k_gsa = (const bf16_t*)a->k_gsa;
  p.v = (const bf16_t*)a->v; p.s = (const bf16_t*)a->s; p.g = (const bf16_t*)a->g;
  p.o = (bf16_t*)a->o;
  p.lse_swa = a->lse_swa; p.lse_gsa = a->lse_gsa;
  p.h0k = a->h0k; p.h0v = a->h0v; p.hkt = a->hkt; p.hvt = a->hvt;
  p.cu = a->cu_seqlens; p.cidx = a->chunk_indices; p.coff = a->chunk_offsets;
  const ScratchPlan sp = plan_call(a);
  char* sc = (char*)a->scratch;
  p.hkT = (bf16_t*)(sc + sp.hkT);
  p.hvc = (bf16_t*)(sc + sp.hvc);
  p.gc = (float*)(sc + sp.gc);
  p.dcum = (float*)(sc + sp.dcum);
  p.hend_k = (float*)(sc + sp.hend_k);
  p.hend_v = (float*)(sc + sp.hend_v);
  p.hseg_k = (float*)(sc + sp.hseg_k);
  p.hseg_v = (float*)(sc + sp.hseg_v);
  p.dtot = (float*)(sc + sp.dtot);
  p.flags = (int*)(sc + sp.flags);
  p.T_tot = a->T_tot; p.N = a->N; p.NT = a->NT; p.HQ = a->HQ; p.H = a->H; p.NG = a->HQ / a->H;
  p.wl = a->wl; p.shift = a->shift; p.scale = a->scale;
  p.seg_sh = sp.seg_sh;
  return p;
}
}  // namespace

int prefill_mfma_impl(const NhaPrefillArgs* a, int phase) {
  const MP p = make_mp(a);
  hipStream_t st = (hipStream_t)a->stream;
  if (a->K == 64) return run_mfma<64>(p, phase, st);
  if (a->K == 128) return run_mfma<128>(p, phase, st);
  return run_mfma<256>(p, phase, st);
}

// The state pass of `a` in the segment form (the backward's): `out` receives the parameter block whose tables it filled --
// segment-local chunk-start states, segment-start states, decays and gate cumsums.
int prefill_mfma_segment_states(const NhaPrefillArgs* a, MP* out) {
  const MP p = *out = make_mp(a);
  hipStream_t st = (hipStream_t)a->stream;
  if (p.NT > 65535) {
    set_error("nha_prefill_bwd(mfma): more than 65535 chunks (%d) in one call", p.NT);
    return NHA_ERR_UNSUPPORTED;
  }
  return a->K == 64 ? run_state_pass<64>(p, true, st) : a->K == 128 ? run_state_pass<128>(p, true, st) : run_state_pass<256>(p, true, st);
}

}  // namespace nha
