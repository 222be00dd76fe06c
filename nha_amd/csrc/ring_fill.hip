// Hand-over of a prompt to a decode ring in one launch (nha_ring_fill; the slicing of nha_fla/models/nha_cache.py:87-91).
//
// Ring slot r of sequence n takes the newest token j of the sequence with j % W == r (zeros where there is none), in all
// four rings at once; the slot states and the token counts are copied beside it.  Rows are moved as 16-byte pieces
// whatever their element type.  Bound: launches -- the bytes are a few MB at most.  As tensor operations (token numbers,
// a gather and a product with the validity per ring, two copies of states) the same hand-over was 22 launches: a prompt of
// 331 tokens through a 32/4-head block of 128 with W = 64 took 351 us per call, of which the host's share of these was the
// largest; with one launch 181 us.
#include "common.h"

namespace nha {
namespace {

struct RingFillP {
  const uint4* src[4];   // window keys, slot keys, values, log gates: [tokens][row]
  uint4* dst[4];         // [N][W][row]
  int np[4];             // 16-byte pieces per row
  const uint4* state[2];
  uint4* state_out[2];
  int64_t ns[2];         // pieces per sequence
  const int32_t* cu;     // [N+1], or NULL: sequences of T tokens
  int32_t* count;
  int64_t tokens;
  int T, W;
};

// grid (W + state workgroups, N)
__global__ __launch_bounds__(256) void ring_fill_kernel(const RingFillP p) {
  const int n = blockIdx.y, W = p.W;
  if ((int)blockIdx.x >= W) {
    const int64_t stride = (int64_t)(gridDim.x - W) * 256;
    for (int x = 0; x < 2; ++x) {
      const uint4* const src = p.state[x] + n * p.ns[x];
      uint4* const dst = p.state_out[x] + n * p.ns[x];
      for (int64_t i = (int64_t)(blockIdx.x - W) * 256 + threadIdx.x; i < p.ns[x]; i += stride) dst[i] = src[i];
    }
    return;
  }
  const int r = blockIdx.x;
  const int64_t start = p.cu ? p.cu[n] : (int64_t)n * p.T;
  const int len = p.cu ? p.cu[n + 1] - p.cu[n] : p.T;
  // the newest token whose number is r modulo W
  const int tok = len - 1 < r ? -1 : len - 1 - (len - 1 - r) % W;
  const bool has = tok >= 0 && start >= 0 && start + tok < p.tokens;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int np = p.np[x];
    const uint4* const src = p.src[x] + (start + tok) * np;
    uint4* const dst = p.dst[x] + ((int64_t)n * W + r) * np;
    for (int i = threadIdx.x; i < np; i += 256) dst[i] = has ? src[i] : make_uint4(0, 0, 0, 0);
  }
  if (r == 0 && threadIdx.x == 0) p.count[n] = len;
}

}  // namespace

int ring_fill_impl(const NhaRingFillArgs* a) {
  RingFillP p;
  for (int x = 0; x < 4; ++x) {
    p.src[x] = (const uint4*)a->src[x];
    p.dst[x] = (uint4*)a->ring[x];
    p.np[x] = a->row_bytes[x] / 16;
  }
  int64_t most = 0;
  for (int x = 0; x < 2; ++x) {
    p.state[x] = (const uint4*)a->state[x];
    p.state_out[x] = (uint4*)a->state_out[x];
    p.ns[x] = a->state_bytes[x] / 16;
    if (p.ns[x] > most) most = p.ns[x];
  }
  p.cu = a->cu_seqlens;
  p.count = a->count;
  p.tokens = a->tokens;
  p.T = a->T;
  p.W = a->W;
  // a state workgroup moves about four pieces per thread of each state
  int64_t sw = (most + 1023) / 1024;
  if (sw > 1024) sw = 1024;
  hipLaunchKernelGGL(ring_fill_kernel, dim3(a->W + (int)sw, a->N), dim3(256), 0, (hipStream_t)a->stream, p);
  NHA_CHECK_LAUNCH("nha_ring_fill");
  return NHA_OK;
}

}  // namespace nha
