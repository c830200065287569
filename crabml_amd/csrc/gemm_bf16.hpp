// gemm_bf16.hpp -- rows x bfloat16 weights on the matrix cores: the prompt-time linear of the hybrid decoder.
//
//   C[row][n] = sum_k A[row][k] W[n][k]     A: bf16 planes, W: bf16 rows, f32 accumulation (v_mfma_f32_16x16x32_bf16)
//
// One plane of A is bf16 arithmetic.  Three planes are a row of f32 numbers cut into its upper, middle and lower eight significand
// bits (split3): every f32 is the exact sum of its planes and every plane times a bf16 weight is exact in f32, so three planes give
// true f32 products with f32 sums -- the weights ARE bf16 numbers -- at a fifth of the time the f32 matrix instruction would take.
//
// Mapping: BM x 128 output tile per workgroup (BM = 256 and 128: eight waves; else four), k in steps of 64.  A step's tiles go from memory
// straight into LDS (global_load_lds, 16 bytes per lane); three or four steps are in LDS or on their way, and a wave waits for the oldest
// only (s_waitcnt vmcnt(n)).  LDS holds rows of 128 bytes whose 16-byte chunks are permuted by (row / 2) % 8 -- on the SOURCE side, the LDS side of the instruction
// being linear -- so that the 16 rows a fragment read touches spread over all 64 banks.  Operands are padded by their owners (k to 64,
// weight rows to 256, activation rows to 256), so the loop has no bounds checks; stores have.  Short launches cut k into pieces (the
// last workgroup of a tile adds them).  Workgroups are dealt to the eight XCDs
// in contiguous runs of the tile order, row tiles fastest: an XCD's L2 keeps the weight tile that its row tiles share.
//
// The row operations around a linear are folded into it.  In: an RMS norm with a single gain is a factor per row, applied to the
// accumulators (the producers leave each row's sum of squares in 64-column pieces); a gain per column is in the planes already.  Out:
// activations by column range, xIELU, a gated unit, soft cap, or the residual add (of one stream or of several that mix), which also
// leaves the new row's bf16 planes and square sums for the next linear.
#pragma once
#include "gemv_bf16.hpp"
#include "lds_dma.hpp"

namespace crabml_hip {

typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

enum {
  GEMM_OUT_ACT_BF16 = 0,   // rows of bf16 (ActRanges)
  GEMM_OUT_ACT_F32 = 1,    // rows of f32 (ActRanges)
  GEMM_OUT_RESIDUAL = 2,   // x += acc (+ add_rows + add_vec); planes of x; square sums
  GEMM_OUT_XIELU = 3,      // planes of xielu(acc)
  GEMM_OUT_SOFTCAP = 4,    // f32 rows
  GEMM_OUT_STREAMS = 5,    // the residual streams take acc (+ bias); planes of gain_next * what the next linear reads; its square sums
  GEMM_OUT_GLU = 6,        // weight rows 2 j, 2 j + 1 are gate j and up j: planes of gelu(gate) * up
};

// an f32 as bf16 planes: 1 plane = rounded to nearest even; 3 planes = upper / middle / lower bits, their sum exact
template <int P>
__device__ __forceinline__ void split_store(float v, unsigned short* p, size_t plane_stride) {
  if constexpr (P == 1) {
    *p = f2bf(v);
  } else {
    const float hi = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) & 0xffff0000u);
    const float r = v - hi;  // exact: the low 16 bits of the significand
    const float mid = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, r) & 0xffff0000u);
    p[0] = (unsigned short)(__builtin_bit_cast(unsigned, hi) >> 16);
    p[plane_stride] = (unsigned short)(__builtin_bit_cast(unsigned, mid) >> 16);
    p[2 * plane_stride] = f2bf(r - mid);
  }
}

// four neighbouring columns at once (p: 8-byte aligned)
template <int P>
__device__ __forceinline__ void split_store4(const float (&v)[4], unsigned short* p, size_t plane_stride) {
  unsigned short t[P][4];
#pragma unroll
  for (int e = 0; e < 4; e++) split_store<P>(v[e], &t[0][e], 4);
#pragma unroll
  for (int i = 0; i < P; i++) __builtin_memcpy(p + i * plane_stride, t[i], 8);
}

// eight of them (p: 16-byte aligned)
template <int P>
__device__ __forceinline__ void split_store8(const float (&v)[8], unsigned short* p, size_t plane_stride) {
  unsigned short t[P][8];
#pragma unroll
  for (int e = 0; e < 8; e++) split_store<P>(v[e], &t[0][e], 8);
#pragma unroll
  for (int i = 0; i < P; i++) {
    i32x4 w;
    __builtin_memcpy(&w, t[i], 16);
    *(i32x4*)(p + i * plane_stride) = w;
  }
}
__device__ __forceinline__ void read8(const float* p, float (&o)[8]) {
  const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + 4);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    o[e] = a[e];
    o[e + 4] = b[e];
  }
}

// One step of 64: TM x TN fragments of products of rows ra + 16 i of the stage at `la` and rows rb + 16 j of the one at `lb`.  LDS rows are 64
// elements, their 16-byte pieces permuted by (row / 2) % 8.  request(d), d < NREQ, asks for a part of a later step: requests are spread over the
// products, because 48 KB a step are 768 cycles of the CU's address path, and issued in a row behind the barrier they left the matrix
// cores idle for 550 of a step's 2150 cycles (256 x 128 tile, 2048 x 11264 x 2048: 138 -> 115 us).
template <typename V, int TM, int TN, int NREQ, typename Mul, typename Req>
__device__ __forceinline__ void tile_step(const unsigned short* la, int ra, const unsigned short* lb, int rb, Mul mul, Req request) {
  constexpr int GR = 2 * TM, SL = TM > 1 ? TM - 1 : 1;
  const int fr = threadIdx.x & 15, fk = threadIdx.x >> 4 & 3;
  V f[2][TN + TM];  // columns, rows
  auto read = [&](int kk, int i) {
    const int r = i < TN ? rb + i * 16 + fr : ra + (i - TN) * 16 + fr;
    f[kk][i] = *(const V*)((i < TN ? lb : la) + r * 64 + (((kk * 4 + fk) ^ ((r >> 1) & 7)) * 8));
  };
#pragma unroll
  for (int i = 0; i < TN + TM; i++) read(0, i);
#pragma unroll
  for (int q = 0; q < GR; q++) {
    const int kk = q / TM, i = q % TM;
#pragma unroll
    for (int j = 0; j < TN; j++) mul(i, j, f[kk][TN + i], f[kk][j]);
    __builtin_amdgcn_sched_barrier(0);
    if (q < SL) {  // the second half's fragments, behind all but the last group of the first
#pragma unroll
      for (int d = (TN + TM) * q / SL; d < (TN + TM) * (q + 1) / SL; d++) read(1, d);
    }
#pragma unroll
    for (int d = NREQ * q / GR; d < NREQ * (q + 1) / GR; d++) request(d);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// S > 1: k is cut into S pieces, one workgroup each.  A workgroup leaves its accumulators (F fragments a thread, NT threads) in ws
// (write-through) and counts itself in; the one that comes last adds all pieces in piece order, whoever it is, and goes on to the epilogue
// (true).  The counter is left at zero.
template <int F, int NT>
__device__ __forceinline__ bool add_pieces(f32x4* acc, int S, int piece, int tile, float* ws, unsigned* tick) {
  constexpr int FRAG = F * 2;  // 8-byte halves of a thread's accumulators
  const int tid = threadIdx.x;
  unsigned long long* base = (unsigned long long*)ws + (size_t)tile * S * NT * FRAG + tid;
  unsigned long long* mine = base + (size_t)piece * NT * FRAG;
#pragma unroll
  for (int i = 0; i < F; i++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const f32x2 v = {acc[i][2 * e], acc[i][2 * e + 1]};
      __hip_atomic_store(mine + (i * 2 + e) * NT, __builtin_bit_cast(unsigned long long, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's write-through stores have been acknowledged
  __shared__ unsigned s_last;
  __syncthreads();
  if (tid == 0) s_last = __hip_atomic_fetch_add(tick + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(S - 1);
  __syncthreads();
  if (!s_last) return false;
  if (tid == 0) __hip_atomic_store(tick + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int i = 0; i < F; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int q = 0; q < S; q++) {
    const unsigned long long* p = base + (size_t)q * NT * FRAG;
#pragma unroll
    for (int i = 0; i < F; i++)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const f32x2 v = __builtin_bit_cast(f32x2, __hip_atomic_load(p + (i * 2 + e) * NT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        acc[i][2 * e] += v[0];
        acc[i][2 * e + 1] += v[1];
      }
  }
  return true;
}

struct GemmBf16 {
  const unsigned short* a = nullptr;  // [planes][rows padded][k]
  size_t a_plane = 0;                 // elements between planes
  const unsigned short* w = nullptr;  // [N padded][k]
  int M = 0, N = 0, K = 0;            // K % 64 == 0
  // row factor (nullable sq): gain (nullable: 1) / sqrt(sum_i sq[row][i] / mean_n + eps)
  const float* sq_in = nullptr;
  int n_sq = 0, mean_n = 1;
  float eps = 0.f;
  const float* gain = nullptr;
  // outputs
  void* out = nullptr;  // ACT / SOFTCAP rows
  int ldo = 0;
  ActRanges act;
  const float* xielu = nullptr;
  float cap = 0.f;
  const float* bias = nullptr;  // [N padded to 8], nullable (ACT, STREAMS)
  float* x = nullptr;           // RESIDUAL; STREAMS: stream 0
  StreamMix sm;
  const float* gain_next = nullptr;  // STREAMS: a gain per column of the next RMS norm
  int ldx = 0;
  const float *add_rows = nullptr, *add_vec = nullptr;
  unsigned short* planes = nullptr;  // RESIDUAL / STREAMS / XIELU / GLU: [planes][rows padded][ldp]
  size_t p_plane = 0;
  int ldp = 0;
  float* sq_out = nullptr;  // [row][n_sq_out]: square sums by 64 columns
  int n_sq_out = 0;
};

// room for k pieces: partial tiles, and a zeroed counter per tile
#define GEMM_TICKS 4096
struct GemmScratch {
  float* partials = nullptr;
  size_t floats = 0;
  unsigned* ticks = nullptr;
};
// rows of a tile and pieces of k for M rows x col_tiles tiles of 128 columns, `steps` steps of 64
struct GemmPlan {
  int bm, S;
};
GemmPlan gemm_plan(int M, int col_tiles, int steps, int n_cu, size_t ws_floats);

// gemm_f16.hip: F16 weights
struct GemmF16 {
  const void* a = nullptr;  // rows of f16, a_stride bytes apart (a multiple of 16)
  size_t a_stride = 0;
  const unsigned short* w[3] = {nullptr, nullptr, nullptr};  // [n][K]
  float* out[3] = {nullptr, nullptr, nullptr};               // [M][n]
  int n[3] = {0, 0, 0};
  int end[3] = {0, 0, 0};  // column tiles up to and with this matrix
  int M = 0, K = 0;
};
// planes: 1 or 3 (GEMM_OUT_ACT_BF16 goes with one, GEMM_OUT_ACT_F32 with three)
void launch_gemm_bf16(crabml_hip_device* dev, crabml_hip_device::ProfRec* rec, int planes, int out, const GemmBf16& g, const GemmScratch& w);

}  // namespace crabml_hip
