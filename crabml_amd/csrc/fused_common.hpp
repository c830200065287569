// fused_common.hpp -- rhs quantizer lanes, weight prefetch, embedding, RMSNorm (+ quantize), q/k/v GEMV + rope + KV append, softmax row
// Part of the fused decode step (fused.hip includes the three fused_*.hpp files once, in order; they are not stand-alone
// translation units: the kernels are launched from fused.hip's host code).
#pragma once
#include "dequant.hpp"
#include "gemv_core.hpp"
#include "kernels.hpp"
#include "prefetch.hpp"
#include "sampler.hpp"
#include <type_traits>

namespace crabml_hip {

// exp_f32_cached (buf_f32.rs:29-35)
__device__ __forceinline__ float exp_cached_f(float x, const unsigned short* __restrict__ table) {
  return h2f(table[f2h(x)]);
}

// ---- the rhs quantizer of matmul_vec, one 32-lane half-wave per 32-element block ------------------------------
// Q81 = false: Q8_0 (buf_q8_0.rs:87-134: d = max|x| / 127, q = trunc(x / d) with the simd cast's NaN -> 0; aux = the
// i32 sum of the block's quants -- exact, derived, used for Q4_0's -8 offset).  Q81 = true: Q8_1 (buf_q8_1.rs:90-129:
// q = trunc(clamp(x / d, -128, 127)) with NaN -> -128, aux = the f16 s = d * sum q).  All 32 lanes of the half-wave
// call it (dead lanes with live = false and v = 0).
struct QLane {
  signed char q;
  unsigned short d;
  int aux;
};
template <bool Q81>
__device__ __forceinline__ QLane quant_lane32(float v, bool live) {
  QLane o;
  const float amax = half_max_f32(fabsf(v));
  const float dd = amax / 127.0f;
  o.d = f2h(dd);
  if constexpr (!Q81) {
    const int qi = rs_f32_as_i32(v / dd);
    o.q = (signed char)(unsigned char)((unsigned)qi & 0xffu);  // `as i8` from i32 wraps
    o.aux = half_sum_i32(live ? (int)o.q : 0);
  } else {
    const float c = fminf(fmaxf(v / dd, -128.0f), 127.0f);  // Rust f32::max / min return the non-NaN operand
    const int qi = (int)c;
    o.q = (signed char)qi;
    const int s = half_sum_i32(live ? qi : 0);
    o.aux = (int)f2h((float)s * dd);
  }
  return o;
}
template <bool Q81>
__device__ __forceinline__ void store_qaux(void* aux, int blk, int v) {
  if constexpr (Q81)
    ((unsigned short*)aux)[blk] = (unsigned short)v;
  else
    ((int*)aux)[blk] = v;
}

// ---- Q8_K planes straight from the kernels that produce the vector ------------------------------------------------------
// A Q8_K super-block is 256 elements and its scale comes from the FIRST element of maximal |x| among them
// (buf_q8_k.rs:84-131), but the producers own less: an attention workgroup one head (head_dim values), a gate/up workgroup
// 32 rows.  Every producer publishes its values as 8-byte {f32, epoch} granules (one write-through store carries data and
// tag), gathers the rest of its super-block from its neighbours' granules (bounded polls), runs the whole block's quantizer
// (q8k_wave_quant: the arithmetic of the stand-alone quantizer launch, bit for bit) and stores the part that is its own.
// The consuming GEMV then only copies finished planes into LDS instead of quantizing the f32 vector in its prologue
// (56 super-blocks per workgroup for ffn_down).  All producers of a super-block are co-resident by construction.
struct Q8KExchange {
  unsigned long long* gran;  // one granule per element of the vector
  const int* serial;         // decode-step serial number (never reset): epoch = serial * nseg + seg + 1
  int* fault;
  int nseg, seg;
};
// called by ONE whole wave.  own: this workgroup's n_own consecutive values (LDS), the first of which is element `first` of
// the vector; n_own divides 256 and is a multiple of 16.  oq / od / obs / oqp: the Q8_K planes of the vector (q | d | bsums | qp).
__device__ __forceinline__ void q8k_exchange_store(const Q8KExchange& ex, const float* own, int first, int n_own, int lane,
                                                   signed char* __restrict__ oq, float* __restrict__ od, short* __restrict__ obs,
                                                   signed char* __restrict__ oqp) {
  const unsigned epoch = (unsigned)(*ex.serial) * (unsigned)ex.nseg + (unsigned)ex.seg + 1u;
  if (n_own < 256) {
    for (int i = lane; i < n_own; i += 64)
      __hip_atomic_store(ex.gran + first + i, ((unsigned long long)epoch << 32) | (unsigned long long)__builtin_bit_cast(unsigned, own[i]),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the granules are on their way before the polls queue up behind them
  }
  const int sb = first >> 8, e0 = sb * 256 + 4 * lane;  // this lane's four elements of the super-block
  const bool mine = e0 >= first && e0 < first + n_own;
  f32x4 v;
  if (mine) {
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = own[e0 - first + i];
  } else {
    unsigned long long g[4];
#pragma unroll
    for (int i = 0; i < 4; i++) g[i] = __hip_atomic_load(ex.gran + e0 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      int tries = 0;
      while ((unsigned)(g[i] >> 32) != epoch && tries < (1 << 21)) {
        __builtin_amdgcn_s_sleep(2);
        g[i] = __hip_atomic_load(ex.gran + e0 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        tries++;
      }
      if ((unsigned)(g[i] >> 32) != epoch) *ex.fault = 1;  // a neighbour never arrived: flagged, not hung
      v[i] = __builtin_bit_cast(float, (unsigned)g[i]);
    }
  }
  const Q8KLane o = q8k_wave_quant(v, lane);
  q8k_store_class_major(oqp + sb * 256, lane, o.packed, mine);
  if (mine) {
    ((unsigned*)oq)[sb * 64 + lane] = o.packed;
    if ((lane & 3) == 0) obs[sb * 16 + (lane >> 2)] = (short)o.quad_sum;
  }
  if (lane == 0 && first == sb * 256) od[sb] = o.d;
}

// ---- embedding lookup: copy_rows_from(token_embed, [token]) (llama2.rs:222-223) ----------------------
__global__ __launch_bounds__(256) void k_embed(const char* __restrict__ w, int dtype, size_t off_scale,
                                               const int* __restrict__ token_d, int dim, float* __restrict__ x) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= dim) return;
  // blockIdx.y: row of a prefill batch (token ids and output rows are consecutive); 0 for a decode step
  x[(size_t)blockIdx.y * dim + i] = dequant_elem(w, dtype, off_scale, (size_t)token_d[blockIdx.y] * dim + i);
}

// ---- rmsnorm * weight -> Q8_0 planes ------------------------------------------------------------------
// rms_norm.rs:33-46 (ordered 32-chunk sums, serial chunk accumulation, true division), arithmetic.rs:57-66
// (x * w), buf_q8_0.rs:87-134 (truncating quantizer).  x itself is left untouched: it is the residual.
// Executed by ONE 1024-thread workgroup (16 waves: 4 per SIMD, so the two IEEE divisions per element
// overlap across waves).  It is pure latency, so every global load (x and the norm weight) is issued up
// front in one batch and kept in registers (NIT values per thread); the ordered chunk sums are taken from
// an LDS copy.  Outputs (q / d / isum) may live in LDS (GEMV prologue) or in global memory.
struct NormLds {  // carved from dynamic LDS: xs[cols] f32 | chunk_sums[cols/32] f32
  float* xs;
  float* chunk_sums;
};
__host__ __device__ inline size_t norm_lds_bytes(int cols) { return (size_t)(cols + cols / 32) * sizeof(float); }

// QUANT = false: the normalized row goes to xn_out as f32 (formats whose rhs is not Q8_0 quantize it afterwards)
// xv, wv: this thread's elements it * 1024 + tid of the row and of the gain (0 past the end); cols <= NIT * 1024, blockDim.x == 1024
template <int NIT, bool QUANT, bool Q81 = false>
__device__ __forceinline__ void norm_quant_regs(const float (&xv)[NIT], const float (&wv)[NIT], int cols, float eps, NormLds L, float* s_rms,
                                                signed char* q, unsigned short* d, void* isum, float* xn_out, int half) {
  const int nchunks = cols / 32;
  const int tid = threadIdx.x;
#pragma unroll
  for (int it = 0; it < NIT; it++) {
    int i = it * 1024 + tid;
    if (i < cols) L.xs[i] = xv[it];
  }
  __syncthreads();
  for (int c = tid; c < nchunks; c += 1024) {
    const f32x4* p = (const f32x4*)(L.xs + c * 32);
    float s = -0.0f, s1 = -0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      f32x4 t = p[j];
      float& a = (half && j >= 4) ? s1 : s;
      a += t[0] * t[0];
      a += t[1] * t[1];
      a += t[2] * t[2];
      a += t[3] * t[3];
    }
    // half (fast mode): chunk = (rows 0..15 in order) + (rows 16..31 in order), the split the wo / ffn_down norm
    // epilogue uses (two workgroups per chunk); otherwise the reference's 32-element scan (rms_norm.rs:35-38)
    L.chunk_sums[c] = half ? s + s1 : s;
  }
  __syncthreads();
  if (tid < 64) {
    // chunk sums are added strictly in chunk order (rms_norm.rs:35-40): wave 0 holds them in registers and
    // v_readlane feeds a single dependent v_add chain.  Lanes past nchunks contribute +0.0 (exact).
    float sum = 0.0f;
    for (int base = 0; base < nchunks; base += 64) {
      float v = base + tid < nchunks ? L.chunk_sums[base + tid] : 0.0f;
      if (half) {
        // fast mode: 64 chunk sums per round through the DPP tree (wave_sum_f32), rounds added in order -- the order of the
        // wo / ffn_down norm epilogue, where a 128-step dependent v_add chain sat between the last arriving granule and the
        // quantizer (0.4 us per hop on MI355X: a dependent f32 add issues every ~8 cycles)
        sum += wave_sum_f32(v);
      } else {
#pragma unroll
        for (int i = 0; i < 64; i++) sum += rl_f(v, i);
      }
    }
    if (tid == 0) *s_rms = sqrtf(sum / (float)cols + eps);
  }
  __syncthreads();
  const float rms = *s_rms;
#pragma unroll
  for (int it = 0; it < NIT; it++) {
    int i = it * 1024 + tid;
    if (it * 1024 < cols) {  // wave-uniform; 32-lane halves are entirely in or out of range (cols % 32 == 0)
      bool live = i < cols;
      float v = live ? (xv[it] / rms) * wv[it] : 0.f;
      if constexpr (!QUANT) {
        if (live) xn_out[i] = v;
        continue;
      }
      const QLane o = quant_lane32<Q81>(v, live);
      if (live) {
        q[i] = o.q;
        if ((tid & 31) == 0) {
          d[i >> 5] = o.d;
          store_qaux<Q81>(isum, i >> 5, o.aux);
        }
      }
    }
  }
}
template <int NIT, bool QUANT, bool Q81 = false>  // cols <= NIT * 1024, blockDim.x == 1024; ends with the outputs written
__device__ __forceinline__ void norm_quant_block(float* __restrict__ x, const float* __restrict__ addv,
                                                 const float* __restrict__ w, int cols, float eps, NormLds L,
                                                 float* s_rms, signed char* q, unsigned short* d, void* isum,
                                                 float* __restrict__ xn_out, int half) {
  const int tid = threadIdx.x;
  float xv[NIT], wv[NIT];
#pragma unroll
  for (int it = 0; it < NIT; it++) {
    int i = it * 1024 + tid;
    xv[it] = i < cols ? x[i] : 0.f;
    wv[it] = i < cols ? w[i] : 0.f;
    // tensor-parallel: the all-reduced wo / ffn_down output is added to the residual stream here
    // (x = matmul_out + x, llama2.rs:266 / :636) and written back
    if (addv != nullptr && i < cols) {
      xv[it] = addv[i] + xv[it];
      x[i] = xv[it];
    }
  }
  norm_quant_regs<NIT, QUANT, Q81>(xv, wv, cols, eps, L, s_rms, q, d, isum, xn_out, half);
}

template <int NIT, bool Q81>
__global__ __launch_bounds__(1024) void k_norm_quant(float* __restrict__ x, const float* __restrict__ addv,
                                                    const float* __restrict__ w, int cols, float eps,
                                                    signed char* __restrict__ q, unsigned short* __restrict__ d,
                                                    void* __restrict__ isum, int half) {
  extern __shared__ float lds[];
  __shared__ float s_rms;
  NormLds L{lds, lds + cols};
  norm_quant_block<NIT, true, Q81>(x, addv, w, cols, eps, L, &s_rms, q, d, isum, nullptr, half);
}
template <int NIT>
__global__ __launch_bounds__(1024) void k_norm_f32(float* __restrict__ x, const float* __restrict__ addv,
                                                  const float* __restrict__ w, int cols, float eps, float* __restrict__ xn, int half) {
  extern __shared__ float lds[];
  __shared__ float s_rms;
  NormLds L{lds, lds + cols};
  norm_quant_block<NIT, false>(x, addv, w, cols, eps, L, &s_rms, nullptr, nullptr, nullptr, xn, half);
}

// ---- the front of a decode step in one launch: sampler's second stage, embedding, first norm, its quantizer -------------
// These were four launches at a step's two ends (combine the arg-max partials, embedding, norm, quantizer of a Q8_K rhs): each is one
// round trip to memory behind 1.7 us of launch.  One workgroup does all of it: every wave combines the partials for itself (two
// requests a lane), so the token is known without a barrier; the row's elements are requested together whatever the table's format is.
// Inside a graph of several steps (run_steps) it runs at the END of a step, for the next one; a graph's first step runs it without the partials.
// With several steps in a graph (run_steps), us a request, before -> after: 57 tokens of the 15M-parameter model in Q8_0 6482 -> 6047, 88 tokens of 8
// layers of the 8B shape in Q4_0 24840 -> 24232.
enum { FRONT_ROW = 0, FRONT_Q8_0 = 1, FRONT_Q8_1 = 2, FRONT_Q8_K = 3, FRONT_SUMS = 4 };  // what is left beside x: nothing, the normed row's planes, sums of squares of 16
struct TokenPick {  // pv == nullptr: the token is *token; logits: the n of them in place of the partials
  const float* logits = nullptr;
  int n = 0;
  const float* pv = nullptr;
  const int* pi = nullptr;
  int nparts = 0, out_cap = 0;
  int *token = nullptr, *pos = nullptr, *step = nullptr, *serial = nullptr;
  unsigned* out = nullptr;
};
struct FrontOut {
  signed char *q = nullptr, *qp = nullptr;  // (qp: class-major copy, Q8_K)
  void *d = nullptr, *aux = nullptr;        // scales; block sums
};
// a thread's elements of the row: QUADS of four, 4096 apart, or one every 1024
template <bool QUADS>
__device__ __forceinline__ int front_elem(int it) {
  return QUADS ? (it >> 2) * 4096 + (int)threadIdx.x * 4 + (it & 3) : it * 1024 + (int)threadIdx.x;
}
template <int NIT, bool QUADS>
__device__ __forceinline__ void embed_row(const char* __restrict__ w, int dtype, size_t off_scale, size_t base, int dim, float (&v)[NIT]) {
  // (one format at a time: with the format's switch inside the loop each element's request waited for the one before it)
  auto all = [&](auto t) {
#pragma unroll
    for (int it = 0; it < NIT; it++) {
      const int i = front_elem<QUADS>(it);
      const float e = dequant_elem(w, decltype(t)::value, off_scale, base + (i < dim ? i : dim - 1));
      v[it] = i < dim ? e : 0.f;
    }
  };
  switch (dtype) {
    case CRABML_HIP_Q4_0: all(std::integral_constant<int, CRABML_HIP_Q4_0>()); break;
    case CRABML_HIP_Q8_0: all(std::integral_constant<int, CRABML_HIP_Q8_0>()); break;
    case CRABML_HIP_Q4_1: all(std::integral_constant<int, CRABML_HIP_Q4_1>()); break;
    case CRABML_HIP_Q4_K: all(std::integral_constant<int, CRABML_HIP_Q4_K>()); break;
    case CRABML_HIP_Q6_K: all(std::integral_constant<int, CRABML_HIP_Q6_K>()); break;
    case CRABML_HIP_F16: all(std::integral_constant<int, CRABML_HIP_F16>()); break;
    case CRABML_HIP_F32: all(std::integral_constant<int, CRABML_HIP_F32>()); break;
    default:
#pragma unroll 1
      for (int it = 0; it < NIT; it++) {
        const int i = front_elem<QUADS>(it);
        v[it] = i < dim ? dequant_elem(w, dtype, off_scale, base + i) : 0.f;
      }
  }
}
// A scan of squares from -0.0 through 4 or 8 lanes of four elements each (last = 3 or 7), handed from lane to lane: the group's last lane has it
__device__ __forceinline__ float quad_square_scan(const f32x4 v, int lane, int last) {
  const f32x4 q = v * v;
  float t = (((-0.0f + q[0]) + q[1]) + q[2]) + q[3];
  for (int k = 1; k <= last; k++) {
    const float u = (((dpp_f<0x111>(t) + q[0]) + q[1]) + q[2]) + q[3];  // (row_shr:1: the lane before goes first)
    t = (lane & last) == k ? u : t;
  }
  return t;
}
// sums of nchunks chunks in norm_quant_regs' order, by every wave for itself
__device__ __forceinline__ float chunk_sums(const float* cs, int nchunks, int lane, int half) {
  float sum = 0.0f;
  for (int base = 0; base < nchunks; base += 64) {
    const float v = base + lane < nchunks ? cs[base + lane] : 0.0f;
    if (half) {
      sum += wave_sum_f32(v);
    } else {
#pragma unroll
      for (int i = 0; i < 64; i++) sum += rl_f(v, i);
    }
  }
  return sum;
}
template <int NIT, int FRONT>
__global__ __launch_bounds__(1024) void k_step_front(const char* __restrict__ table, int dtype, size_t off_scale, TokenPick pick, int dim, float* __restrict__ x,
                                                     const float* __restrict__ wn, float eps, FrontOut o, int half) {
  constexpr bool QUADS = FRONT != FRONT_ROW;  // (rows of whole chunks)
  __shared__ float s_pick[16], s_chunks[NIT * 32];
  __shared__ int s_pick_at[16];
  const int tid = threadIdx.x, lane = tid & 63;
  float xv[NIT];
  f32x4 wv[NIT / 4];
  if constexpr (QUADS && FRONT != FRONT_SUMS) {
#pragma unroll
    for (int j = 0; j < NIT / 4; j++) wv[j] = ((const f32x4*)wn)[j * 4096 + tid * 4 < dim ? j * 1024 + tid : 0];
  }
  int token;
  if (pick.pv != nullptr) {
    float bv = -INFINITY;
    int bi = -1;
    if (pick.logits != nullptr) {
      bi = argmax_row(pick.logits, pick.n, s_pick, s_pick_at);
    } else {
      for (int i = lane; i < pick.nparts; i += 64) argmax_combine(bv, bi, pick.pv[i], pick.pi[i]);
      argmax_wave(bv, bi);
    }
    token = bi;
    if (tid == 0) {
      *pick.token = bi;
      const int st = *pick.step;
      if (st < pick.out_cap) pick.out[st] = (unsigned)bi;
      *pick.step = st + 1;
      *pick.pos = *pick.pos + 1;
      *pick.serial = *pick.serial + 1;
    }
  } else {
    token = *pick.token;
  }
  embed_row<NIT, QUADS>(table, dtype, off_scale, (size_t)token * dim, dim, xv);
  if constexpr (!QUADS) {
#pragma unroll
    for (int it = 0; it < NIT; it++)
      if (it * 1024 + tid < dim) x[it * 1024 + tid] = xv[it];
    return;
  }
  f32x4 v[NIT / 4];
#pragma unroll
  for (int j = 0; j < NIT / 4; j++) {
    const int i = j * 1024 + tid;
    v[j] = f32x4{xv[4 * j], xv[4 * j + 1], xv[4 * j + 2], xv[4 * j + 3]};
    if (i * 4 < dim) ((f32x4*)x)[i] = v[j];
    const float t = quad_square_scan(v[j], lane, half || FRONT == FRONT_SUMS ? 3 : 7);
    if constexpr (FRONT == FRONT_SUMS) {  // (the halves of norm_quant_regs' chunks, as k_kq_res leaves them)
      if ((lane & 3) == 3 && i * 4 < dim) ((float*)o.d)[i >> 2] = t;
    } else {
      const float low = dpp_f<0x114>(t);  // (row_shr:4: rows 0..15's)
      if ((lane & 7) == 7 && i * 4 < dim) s_chunks[i >> 3] = half ? low + t : t;
    }
  }
  if constexpr (FRONT == FRONT_SUMS) return;
  __syncthreads();
  const float rms = sqrtf(chunk_sums(s_chunks, dim / 32, lane, half) / (float)dim + eps);
#pragma unroll
  for (int j = 0; j < NIT / 4; j++) {
    const int i = j * 1024 + tid;
    if (j * 4096 + (tid & ~63) * 4 >= dim) break;  // (wave-uniform)
#pragma unroll
    for (int e = 0; e < 4; e++) v[j][e] = (v[j][e] / rms) * wv[j][e];
    if constexpr (FRONT == FRONT_Q8_K) {
      const int sb = i >> 6;
      const Q8KLane k = q8k_wave_quant(v[j], lane);
      ((unsigned*)o.q)[i] = k.packed;
      q8k_store_class_major(o.qp + sb * 256, lane, k.packed);
      if ((lane & 3) == 0) ((short*)o.aux)[i >> 2] = (short)k.quad_sum;
      if (lane == 0) ((float*)o.d)[sb] = k.d;
    } else {
      const QLane4 k = quant_quad8<FRONT == FRONT_Q8_1>(v[j]);
      if (i * 4 >= dim) continue;  // (whole chunks)
      ((unsigned*)o.q)[i] = k.packed;
      if ((lane & 7) == 0) {
        ((unsigned short*)o.d)[i >> 3] = k.d;
        store_qaux<FRONT == FRONT_Q8_1>(o.aux, i >> 3, k.aux);
      }
    }
  }
}

// batched prefill: one workgroup per row of x (rows, cols) -> xn (rows, cols)
template <int NIT>
__global__ __launch_bounds__(1024) void k_norm_f32_rows(float* __restrict__ x, const float* __restrict__ w, int cols, float eps,
                                                       float* __restrict__ xn, int half) {
  extern __shared__ float lds[];
  __shared__ float s_rms;
  NormLds L{lds, lds + cols};
  norm_quant_block<NIT, false>(x + (size_t)blockIdx.x * cols, nullptr, w, cols, eps, L, &s_rms, nullptr, nullptr, nullptr,
                               xn + (size_t)blockIdx.x * cols, half);
}

// ---- QKV epilogue: rope (rope.rs:47-63) + q scale (llama2.rs:565) + KV append (concatenate.rs:172-204) ---
struct QkvEpi {
  float* q_out;       // (n_heads * hd) f32, roped and scaled
  void* kc;           // K cache of this layer [n_kv][seq_cap][hd]
  void* vc;
  const float* rope;  // [seq_cap][npairs][2] (cos, sin)
  const int* pos_d;
  float scale;        // 1 / sqrt(hd)
  int dim, kv_dim, hd, rope_dim, npairs, seq_cap, kv16;
};

// position + rotation for the pair starting at row0, loaded early (before the weight stream is consumed)
struct QkvPre {
  int pos;
  float c, s;
  bool rot;
};
__device__ __forceinline__ QkvPre qkv_preload(const QkvEpi& e, int row0, int row_of_batch = 0) {
  QkvPre p;
  p.pos = *e.pos_d + row_of_batch;
  p.c = 1.f;
  p.s = 0.f;
  p.rot = false;
  if (row0 < e.dim + e.kv_dim) {
    const int i = (row0 < e.dim ? row0 : row0 - e.dim) % e.hd;
    if (i < e.rope_dim) {
      const float* cs = e.rope + ((size_t)p.pos * e.npairs + (i >> 1)) * 2;
      p.c = cs[0];
      p.s = cs[1];
      p.rot = true;
    }
  }
  return p;
}
// the same without a load inside a branch (the rotation of a clamped pair is fetched unconditionally and ignored where `rot` is
// false): a loaded value that leaves a lane-predicated region is copied at its end, i.e. waited for on the spot -- a memory round
// trip in front of the wave's first weight request
__device__ __forceinline__ QkvPre qkv_preload_nb(const QkvEpi& e, int row0) {
  QkvPre p;
  p.pos = *e.pos_d;
  const int i = (row0 < e.dim ? row0 : row0 - e.dim) % e.hd;
  p.rot = row0 < e.dim + e.kv_dim && i < e.rope_dim;
  const float* cs = e.rope + ((size_t)p.pos * e.npairs + (p.rot ? (i >> 1) : 0)) * 2;
  p.c = cs[0];
  p.s = cs[1];
  return p;
}
__device__ __forceinline__ void qkv_epilogue(const QkvEpi& e, const QkvPre& pre, int row0, float s0, float s1) {
  const int pos = pre.pos;
  if (row0 < e.dim + e.kv_dim) {  // q or k: rotate the (even, odd) pair
    const int i = (row0 < e.dim ? row0 : row0 - e.dim) % e.hd;
    float r0 = s0, r1 = s1;
    if (pre.rot) {
      float c = pre.c, s = pre.s;
      r0 = s0 * c - s1 * s;
      r1 = s0 * s + s1 * c;
    }
    if (row0 < e.dim) {
      e.q_out[row0] = r0 * e.scale;
      e.q_out[row0 + 1] = r1 * e.scale;
    } else {
      const int kr = row0 - e.dim;
      const size_t o = ((size_t)(kr / e.hd) * e.seq_cap + pos) * e.hd + i;
      if (e.kv16) {
        ((unsigned short*)e.kc)[o] = f2h(r0);
        ((unsigned short*)e.kc)[o + 1] = f2h(r1);
      } else {
        ((float*)e.kc)[o] = r0;
        ((float*)e.kc)[o + 1] = r1;
      }
    }
  } else {
    const int vr = row0 - e.dim - e.kv_dim;
    const size_t o = ((size_t)(vr / e.hd) * e.seq_cap + pos) * e.hd + (vr % e.hd);
    if (e.kv16) {
      ((unsigned short*)e.vc)[o] = f2h(s0);
      ((unsigned short*)e.vc)[o + 1] = f2h(s1);
    } else {
      ((float*)e.vc)[o] = s0;
      ((float*)e.vc)[o + 1] = s1;
    }
  }
}

struct Planes {
  const i32x4* q;
  const unsigned short* d;
};
// a Q6_K matrix standing in for one of a Q4_K layer's (llama.cpp *_K_M mixes): base = nullptr means "not used"
struct Planes6 {
  const char* base;
  size_t off_qh;
};

// DEFER: the rhs planes come from a hop-free ffn_down launch -- the row dots are multiplied by 1 / rms (RmsTail, gemv_core.hpp)
template <int FMT, bool DEFER = false>
__global__ __launch_bounds__(128) void k_qkv(Planes wq, Planes wk, Planes wv, typename ActOf<FMT>::type act, int nb, QkvEpi e,
                                             Planes6 wv6, RmsTail rt, int upfront = 0) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + wave_in_wg();
  const int row0 = wave * 2;
  const int total = e.dim + 2 * e.kv_dim;
  if (row0 >= total) return;
  Planes w;
  int local, m;
  if (row0 < e.dim) {
    w = wq; local = row0; m = e.dim;
  } else if (row0 < e.dim + e.kv_dim) {
    w = wk; local = row0 - e.dim; m = e.kv_dim;
  } else {
    w = wv; local = row0 - e.dim - e.kv_dim; m = e.kv_dim;
  }
  QkvPre pre{};
  RmsReq rq{0.f, 0.f};
  if constexpr (DEFER) {
    // (every lane loads the pair's rotation -- one address -- instead of lane 0 alone: with the chunk sums requested next to it, a
    // load inside a lane-predicated branch would make the wave wait for all of them before its first weight request)
    pre = qkv_preload_nb(e, row0);
    rq = rms_request(rt, lane);
  } else {
    if (lane == 0) pre = qkv_preload(e, row0);
  }
  float acc[2];
  bool done = false;
  if constexpr (FMT == CRABML_HIP_Q4_K) {
    if (wv6.base != nullptr && row0 >= e.dim + e.kv_dim) {  // the V rows of this layer are Q6_K (wave-uniform)
      rows_partial_q6k<2>(wv6.base, wv6.off_qh, act, local, m, nb, lane, acc);
      done = true;
    }
  }
  float inv_rms = 1.0f;
  if constexpr (DEFER && FMT != CRABML_HIP_Q4_K) {
    if (upfront && nb * BlockFmt<FMT>::UNITS == 128)
      inv_rms = rows_partial_rms_128<FMT, 2>(w.q, w.d, act, local, m, nb, lane, acc, rt, rq);
    else
      inv_rms = rows_partial_rms<FMT, 2>(w.q, w.d, act, local, m, nb, lane, acc, rt, rq);
  } else {
    if constexpr (FMT != CRABML_HIP_Q4_K) {
      if (!done && upfront && (nb * BlockFmt<FMT>::UNITS) % 128 == 0) {
        rows_partial_2step<FMT, 2>(w.q, w.d, act, local, m, nb, lane, acc);
        done = true;
      }
    }
    if (!done) rows_dot<FMT, 2>(w.q, w.d, act, local, m, nb, lane, acc);
  }
  float s0 = wave_sum_f32(acc[0]), s1 = wave_sum_f32(acc[1]);
  if constexpr (DEFER) {
    s0 *= inv_rms;
    s1 *= inv_rms;
  }
  if (lane == 0) qkv_epilogue(e, pre, row0, s0, s1);
}
// strict order (CRABML_HIP_FLAG_STRICT_ORDER, Q4_0 / Q8_0 / Q4_1 layers): the same launch with the block terms parked in LDS and
// added in block order by one lane per row (rows_terms / ordered_sum, gemv_core.hpp) -- q, k and v rows bit-identical to the scalar
// loops of the reference, then the same epilogue.  Workgroup = 4 waves x one (even, odd) row pair; dynamic LDS = 8 * nt floats.
template <int FMT>
__global__ __launch_bounds__(256) void k_qkv_ord(Planes wq, Planes wk, Planes wv, typename ActOf<FMT>::type act, int nb, QkvEpi e) {
  extern __shared__ __attribute__((aligned(16))) float ord_terms[];
  const int lane = threadIdx.x & 63, wv_i = wave_in_wg();
  const int wave = blockIdx.x * (blockDim.x >> 6) + wv_i;
  const int row0 = wave * 2;
  const int total = e.dim + 2 * e.kv_dim;
  if (row0 >= total) return;
  Planes w;
  int local, m;
  if (row0 < e.dim) {
    w = wq; local = row0; m = e.dim;
  } else if (row0 < e.dim + e.kv_dim) {
    w = wk; local = row0 - e.dim; m = e.kv_dim;
  } else {
    w = wv; local = row0 - e.dim - e.kv_dim; m = e.kv_dim;
  }
  QkvPre pre{};
  if (lane == 0) pre = qkv_preload(e, row0);
  float s = 0.0f;
  const int nt = (nb + 3) & ~3;
  float* T = ord_terms + (size_t)wv_i * 2 * nt;
  rows_terms<FMT, 2, typename ActOf<FMT>::type, true>(w.q, w.d, act, local, m, nb, lane, T, nt);
  __builtin_amdgcn_wave_barrier();
  if (lane < 2) s = ordered_sum(T + lane * nt, nb);
  const float s1 = __shfl(s, 1, 64);
  if (lane == 0) qkv_epilogue(e, pre, row0, s, s1);
}
// strict mode: the three GEMVs ran in scalar order into tmp[dim + 2 kv_dim]; apply the same epilogue
__global__ __launch_bounds__(256) void k_qkv_epi(const float* __restrict__ tmp, QkvEpi e) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  int total = (e.dim + 2 * e.kv_dim) / 2;
  if (p < total) qkv_epilogue(e, qkv_preload(e, 2 * p), 2 * p, tmp[2 * p], tmp[2 * p + 1]);
}

// batched prefill: the three GEMMs wrote qb (B, dim), kb / vb (B, kv_dim); row r is position *pos_d + r
__global__ __launch_bounds__(256) void k_qkv_epi_rows(const float* __restrict__ qb, const float* __restrict__ kb,
                                                     const float* __restrict__ vb, QkvEpi e) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (p >= (e.dim + 2 * e.kv_dim) / 2) return;
  const int row0 = 2 * p;
  const float* src = row0 < e.dim              ? qb + (size_t)r * e.dim + row0
                     : row0 < e.dim + e.kv_dim ? kb + (size_t)r * e.kv_dim + (row0 - e.dim)
                                               : vb + (size_t)r * e.kv_dim + (row0 - e.dim - e.kv_dim);
  QkvEpi er = e;
  er.q_out = e.q_out + (size_t)r * e.dim;
  qkv_epilogue(er, qkv_preload(e, row0, r), row0, src[0], src[1]);
}

// softmax.rs:36-54 over scores[0..seq) in LDS, in place, by a workgroup of NW waves (4 or 16): max, exp through the f16
// table, row sum sequential up to 1024 positions (bit-exact; at every length when seq_sum is set) and a block tree beyond,
// true division.  F16: the
// probabilities are then rounded to f16 (quantize_f32_f16 of the lhs, batch_matmul.rs:39).  Ends with a barrier.
// The tree is defined on 256 partial sums (partial v = positions v, v + 256, ... in order) whatever NW is: 16 waves share
// the max / exp / division passes (the long-context softmax kernel), the sums are the 4-wave kernel's bit for bit.
// s_red: NW floats.
// seq_sum: the row sum stays sequential at ANY length (the strict-order device: softmax.rs:43-48 is one scalar loop; the block
// tree beyond 1024 positions is the fast kernels' re-association, pinned in tests/helpers.FAST_TOL)
template <bool F16, int NW = 4>
__device__ __forceinline__ void softmax_row(float* scores, int seq, const unsigned short* __restrict__ exp_tab, float* s_red,
                                            float* s_val_p, bool seq_sum = false) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int BD = NW * 64;
  float mx = -INFINITY;
  for (int t = tid; t < seq; t += BD) mx = fmaxf(mx, scores[t]);
  mx = wave_max_f32(mx);
  if (lane == 0) s_red[wave] = mx;
  __syncthreads();
  mx = s_red[0];
#pragma unroll
  for (int w = 1; w < NW; w++) mx = fmaxf(mx, s_red[w]);
  __syncthreads();
  float part = 0.0f;
  {
    // the table lookups are independent global gathers: 8 (4) in flight per thread (long rows), summed in t order
    int t = tid;
    for (; t + 7 * BD < seq; t += 8 * BD) {
      float ev[8];
#pragma unroll
      for (int u = 0; u < 8; u++) ev[u] = exp_cached_f(scores[t + u * BD] - mx, exp_tab);
#pragma unroll
      for (int u = 0; u < 8; u++) {
        scores[t + u * BD] = ev[u];
        part += ev[u];
      }
    }
    for (; t + 3 * BD < seq; t += 4 * BD) {
      float ev[4];
#pragma unroll
      for (int u = 0; u < 4; u++) ev[u] = exp_cached_f(scores[t + u * BD] - mx, exp_tab);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        scores[t + u * BD] = ev[u];
        part += ev[u];
      }
    }
    for (; t < seq; t += BD) {
      float ev = exp_cached_f(scores[t] - mx, exp_tab);
      scores[t] = ev;
      part += ev;
    }
  }
  __syncthreads();
  if (seq <= 1024 || seq_sum) {
    if (tid < 64) {
      // sequential row sum (softmax.rs:43-48) without an LDS round trip per add: wave 0 holds 64 values per
      // pass in registers and v_readlane feeds one dependent v_add chain; lanes past `seq` add +0.0 (exact)
      float sum = 0.0f;
      for (int base = 0; base < seq; base += 64) {
        float v = base + tid < seq ? scores[base + tid] : 0.0f;
#pragma unroll
        for (int i = 0; i < 64; i++) sum += rl_f(v, i);
      }
      if (tid == 0) *s_val_p = sum;
    }
  } else {
    if constexpr (NW != 4) {  // the 256 partial sums of the 4-wave tree, from the exponentials in LDS
      part = 0.0f;
      if (tid < 256)
        for (int t = tid; t < seq; t += 256) part += scores[t];
    }
    if (NW == 4 || tid < 256) {
      part = wave_sum_f32(part);
      if (lane == 0) s_red[wave] = part;
    }
    __syncthreads();
    if (tid == 0) *s_val_p = (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
  }
  __syncthreads();
  const float sum = *s_val_p;
  for (int t = tid; t < seq; t += BD) {
    float pv = scores[t] / sum;
    scores[t] = F16 ? h2f(f2h(pv)) : pv;  // quantize_f32_f16 of the lhs (batch_matmul.rs:39), done once
  }
  __syncthreads();
}

}  // namespace crabml_hip
