// sampler.hpp -- the greedy sampler's first stage, shared by the llama step (fused_ffn.hpp) and the hybrid decoder's
// (hybrid_step.hpp): Iterator::max_by keeps the LAST maximum (sampler.rs:109-116).
// ARGMAX_BLOCKS workgroups per row of logits, each over a contiguous slice; a second launch combines and advances.
#pragma once
#include "devutil.hpp"

namespace crabml_hip {

#define ARGMAX_BLOCKS 128
__device__ __forceinline__ void argmax_combine(float& cv, int& ci, float ov, int oi) {
  // keep the later index among equal maxima; an index of -1 means "empty"
  bool take = oi >= 0 && (ci < 0 || ov > cv || (!(cv > ov) && oi > ci));
  if (take) {
    cv = ov;
    ci = oi;
  }
}
__device__ __forceinline__ void argmax_wave(float& v, int& i) {  // over the 64 lanes; every lane gets it
  argmax_combine(v, i, dpp_f<0xB1>(v), dpp_i<0xB1>(i));
  argmax_combine(v, i, dpp_f<0x4E>(v), dpp_i<0x4E>(i));
  argmax_combine(v, i, dpp_f<0x141>(v), dpp_i<0x141>(i));
  argmax_combine(v, i, dpp_f<0x140>(v), dpp_i<0x140>(i));
  float bv = rl_f(v, 0);
  int bi = __builtin_amdgcn_readlane(i, 0);
#pragma unroll
  for (int r = 16; r < 64; r += 16) argmax_combine(bv, bi, rl_f(v, r), __builtin_amdgcn_readlane(i, r));
  v = bv;
  i = bi;
}
// The whole row of logits by one workgroup of 1024 (the front of the next step), in rounds of 32768: up to four of them are shorter than a launch of partials
// in front of it.  Us, partials and front / front: 32000 logits 4.6 + 4.7 / 5.5 (width 288), 128256 4.8 + 5.7 / 9.8 (width 4096).  sv, si: LDS, 16 each; every thread gets the index (-1: an empty row).
#define ARGMAX_ONE 131072
__device__ __forceinline__ int argmax_row(const float* __restrict__ logits, int n, float* sv, int* si) {
  constexpr int U = 8;
  const int tid = threadIdx.x, n4 = n / 4;
  float bv = -INFINITY;
  int bi = -1;
  for (int i0 = 0; i0 < n4; i0 += U * 1024) {
    f32x4 q[U];
#pragma unroll
    for (int u = 0; u < U; u++) q[u] = ((const f32x4*)logits)[i0 + u * 1024 + tid < n4 ? i0 + u * 1024 + tid : n4 - 1];
#pragma unroll
    for (int u = 0; u < U; u++) {  // (ascending indices: whatever is not smaller takes the place.  The last four once more past the end change nothing)
      const int i = (i0 + u * 1024 + tid < n4 ? i0 + u * 1024 + tid : n4 - 1) * 4;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const bool take = !(bv > q[u][e]);
        bv = take ? q[u][e] : bv;
        bi = take ? i + e : bi;
      }
    }
  }
  if (tid < n % 4) argmax_combine(bv, bi, logits[n4 * 4 + tid], n4 * 4 + tid);
  argmax_wave(bv, bi);
  if ((tid & 63) == 0) {
    sv[tid >> 6] = bv;
    si[tid >> 6] = bi;
  }
  __syncthreads();
  bv = sv[tid & 15];
  bi = si[tid & 15];
  argmax_wave(bv, bi);
  return bi;
}
// base: global index of logits[0] (a vocabulary shard of a tensor-parallel classifier; 0 otherwise).  blockIdx.y: row of a batch
// (row_stride floats apart; its partials follow the previous row's)
static __global__ __launch_bounds__(256) void k_argmax_partial(const float* __restrict__ logits, int n, float* __restrict__ pv,
                                                        int* __restrict__ pi, int base, int row_stride) {
  logits += (size_t)blockIdx.y * row_stride;
  pv += blockIdx.y * gridDim.x;
  pi += blockIdx.y * gridDim.x;
  __shared__ float sv[4];
  __shared__ int si[4];
  const int per = (n + gridDim.x - 1) / gridDim.x;
  const int lo = blockIdx.x * per, hi = min(n, lo + per);
  float bv = -INFINITY;
  int bi = -1;
  for (int i = lo + threadIdx.x; i < hi; i += blockDim.x) argmax_combine(bv, bi, logits[i], base + i);
  argmax_wave(bv, bi);
  if ((threadIdx.x & 63) == 0) {
    sv[threadIdx.x >> 6] = bv;
    si[threadIdx.x >> 6] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; w++) argmax_combine(bv, bi, sv[w], si[w]);
    pv[blockIdx.x] = bv;
    pi[blockIdx.x] = bi;
  }
}

}  // namespace crabml_hip
