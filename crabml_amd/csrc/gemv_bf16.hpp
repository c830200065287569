// gemv_bf16.hpp -- bfloat16 weight rows x f32 activations for up to 8 rows of the rhs at a time, with the neighbouring row
// operations folded into its two ends: the decode-time linear of the hybrid decoder (hybrid_step.hpp), and matmul_vec on BF16.
//
// Mapping: a wave owns R consecutive output rows and strides k 512 elements at a time (8 per lane = one aligned 16-byte request per
// row); the rhs rows sit in LDS as f32 in two half-octet planes, so the two ds_read_b128 a lane needs are contiguous across the wave.
// Weights become f32 by a shift / mask, products and sums are f32 fmas: the rhs is never rounded.  The weight requests of a block
// of steps go out before the activations are staged (the first block) or while the previous block is multiplied.  One pass over the
// weights serves NB rhs rows; more rows are further grid rows (blockIdx.y) that hit the same weights in L2 / Infinity Cache.
#pragma once
#include <type_traits>

#include "devutil.hpp"
#include "kernels.hpp"

namespace crabml_hip {

// what happens to an rhs row on the way in
enum {
  GEMV_IN_PLAIN = 0,
  GEMV_IN_RMS = 1,    // the row is RMS-normalized with a single gain.  The row factor is taken from the staged row itself and
                      // applied to the finished dots: W (s x) = s (W x)
  GEMV_IN_SPLIT = 2,  // elements from k_split on still want their RMS normalization; their sum of squares arrives in pieces (ss)
  GEMV_IN_RMSV = 3,   // GEMV_IN_RMS with a gain per element (gain: K numbers), applied while the row is staged
  // the matrix-core form with one plane: rows that their producer left as bf16 (x16)
  GEMV_IN_BF16 = 4,
  GEMV_IN_BF16_RMS = 5,    // times gain (nullable: 1) over the root mean square, its sum of squares in pieces (ss); gains per element are in x16
  GEMV_IN_BF16_SPLIT = 6,  // GEMV_IN_SPLIT: the dots of the elements from k_split on are normalized
};
// what happens to a dot product on the way out
enum {
  GEMV_OUT_STORE = 0,
  GEMV_OUT_ACT = 1,      // (+ bias) column ranges with their own activation (ActRanges)
  GEMV_OUT_RESIDUAL = 2, // out += dot (+ add_rows[b] + add_vec)
  GEMV_OUT_XIELU = 3,    // xielu(dot)
  GEMV_OUT_SOFTCAP = 4,  // cap * tanh(dot / cap)
  GEMV_OUT_STREAMS = 5,  // (+ bias) into the residual streams; what the next linear reads goes to u
  GEMV_OUT_GLU = 6,      // weight rows 2 j, 2 j + 1 are gate j and up j: out[j] = gelu(gate) * up
};
enum { ACT_NONE = 0, ACT_SIGMOID = 1, ACT_SILU = 2 };
struct ActRanges {  // columns [end[i-1], end[i]) take activation kind[i]
  int end[4] = {0, 0, 0, 0};
  int kind[4] = {0, 0, 0, 0};
};

// Residual streams: a sublayer's result y turns the n streams x_s into x_t = sum_s mix[s][t] x_s + out[t] y, and the next linear reads
// u = sum_t in[t] x_t.  All of it is local to an element, so it is the epilogue of the sublayer's last linear.
#define HC_MAX 8
#define HC_ROW (HC_MAX + 1)
struct StreamMix {
  int n = 0;
  size_t stride = 0;            // floats between the streams
  const float* coef = nullptr;  // [HC_MAX][HC_ROW]: row t = mix[0 .. HC_MAX)[t], out[t]; zeros from n on, both ways
  const float* in = nullptr;    // [HC_MAX]: of the sublayer that comes next
};
// (constant address space: scalar loads, which no store can be taken to change)
typedef const float __attribute__((address_space(4))) const_f32;
// x: an element (or a vector of neighbours) of stream 0
template <typename V>
__device__ __forceinline__ void stream_load(const StreamMix& m, const float* x, V (&old)[HC_MAX]) {
  // (four at a time without a branch each -- past the last stream the first one again, with a zero coefficient)
#pragma unroll
  for (int s = 0; s < 4; s++) old[s] = *(const V*)(x + (s < m.n ? s : 0) * m.stride);
#pragma unroll
  for (int s = 4; s < HC_MAX; s++) old[s] = V{};
  if (m.n > 4) {
#pragma unroll
    for (int s = 4; s < HC_MAX; s++) old[s] = *(const V*)(x + (s < m.n ? s : 0) * m.stride);
  }
}
template <typename V>
__device__ __forceinline__ V stream_apply(const StreamMix& m, float* x, const V (&old)[HC_MAX], V y) {
  const_f32 *coef = (const_f32*)(size_t)m.coef, *in = (const_f32*)(size_t)m.in;
  V u = V{};
  if (m.n <= 4) {  // (all coefficients in one go)
    V v[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      v[t] = coef[t * HC_ROW + HC_MAX] * y;
#pragma unroll
      for (int s = 0; s < 4; s++) v[t] += coef[t * HC_ROW + s] * old[s];
      u += in[t] * v[t];
    }
#pragma unroll
    for (int t = 0; t < 4; t++)
      if (t < m.n) *(V*)(x + t * m.stride) = v[t];
    return u;
  }
#pragma unroll 1
  for (int t = 0; t < m.n; t++) {
    const_f32* c = coef + t * HC_ROW;
    V v = c[HC_MAX] * y;
#pragma unroll
    for (int s = 0; s < HC_MAX; s++) v += c[s] * old[s];
    *(V*)(x + t * m.stride) = v;
    u += in[t] * v;
  }
  return u;
}

struct GemvBf16 {
  const unsigned short* w = nullptr;  // [N][ldw]
  const float* x = nullptr;           // [nb][ldx]
  const unsigned short* x16 = nullptr;  // GEMV_IN_BF16*: the same as bf16
  float* out = nullptr;                 // [nb][ldo]
  // on the matrix cores (nullable): where the results go as bf16 -- XIELU, GLU: instead; RESIDUAL, STREAMS: what the next linear reads, times
  // gain_out (nullable) and with its square sums by 16 columns
  unsigned short* out16 = nullptr;
  const float* gain_out = nullptr;
  float* ss_out = nullptr;  // [nb][ld_ss_out]
  int ld_ss_out = 0;
  int N = 0, K = 0, ldw = 0, ldx = 0, ldo = 0, nb = 1;  // K % 8 == 0
  // GEMV_IN_RMS: elements the mean is over, eps, the gain (device); GEMV_IN_SPLIT: the same for the tail, with n_ss pieces of ss[b][ld_ss]
  // (GEMV_IN_BF16_RMS: such pieces too)
  int mean_n = 1;
  float eps = 0.f;
  const float* gain = nullptr;
  int k_split = 0, n_ss = 0, ld_ss = 0;  // (ld_ss: whole fours)
  const float* ss = nullptr;
  ActRanges act;
  const float* xielu = nullptr;  // {softplus(p), 1/2 + softplus(q)}
  const float *add_rows = nullptr, *add_vec = nullptr;
  int ld_add = 0;
  float cap = 0.f;
  const float* bias = nullptr;  // [N], nullable (ACT, STREAMS)
  bool resident = false;  // the weights of all linears that run in turn fit a cache: they are read so that they stay in it (else nontemporal)
  StreamMix sm;                 // STREAMS: out = stream 0, u[b][ldo] = what the next linear reads
  float* u = nullptr;
  // a k shared by two workgroups of the batched linear: their sums as {value, launch} granules [tiles][2][256], and arrivals [tiles][4], two a launch, zero at first
  unsigned long long* half = nullptr;
  unsigned* meet = nullptr;
};

__device__ __forceinline__ float act_sigmoid(float z) { return 1.0f / (1.0f + __expf(-z)); }
__device__ __forceinline__ float act_apply(float z, int kind) {
  if (kind == ACT_NONE) return z;
  const float s = act_sigmoid(z);
  return kind == ACT_SILU ? z * s : s;
}
__device__ __forceinline__ float act_ranges(float z, int col, const ActRanges& a) {
  const int kind = col < a.end[0] ? a.kind[0] : col < a.end[1] ? a.kind[1] : col < a.end[2] ? a.kind[2] : a.kind[3];
  return act_apply(z, kind);
}
// e^z - 1 - z for z <= 0 without the cancellation near zero: its own series below 1/4
__device__ __forceinline__ float exp_minus_line(float z) {
  if (z > -0.25f) {
    float s = 1.0f / 40320.0f;
    s = __builtin_fmaf(s, z, 1.0f / 5040.0f);
    s = __builtin_fmaf(s, z, 1.0f / 720.0f);
    s = __builtin_fmaf(s, z, 1.0f / 120.0f);
    s = __builtin_fmaf(s, z, 1.0f / 24.0f);
    s = __builtin_fmaf(s, z, 1.0f / 6.0f);
    s = __builtin_fmaf(s, z, 0.5f);
    return s * z * z;
  }
  return __expf(z) - 1.0f - z;
}
__device__ __forceinline__ float xielu_apply(float z, float right, float left) {
  const float curved = z > 0.0f ? right * z * z : left * exp_minus_line(z);
  return __builtin_fmaf(0.5f, z, curved);
}
// z / 2 (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3))), the bracket's half being a logistic function of twice the argument
__device__ __forceinline__ float gelu_tanh(float z) {
  const float t = 1.5957691216057308f * __builtin_fmaf(0.044715f * z, z * z, z);
  return z / (1.0f + __expf(-t));
}
__device__ __forceinline__ float soft_cap(float z, float cap) { return cap > 0.0f ? cap * tanhf(z / cap) : z; }

// GEMV_OUT_RESIDUAL: what the thread that will have (row, b) needs, requested ahead of the products
struct ResidualElem {
  float old = 0.f, rows = 0.f, vec = 0.f;
};
__device__ __forceinline__ void residual_load(const GemvBf16& a, int row, int b, ResidualElem& e) {
  e.old = a.out[(size_t)b * a.ldo + row];
  if (a.add_rows) e.rows = a.add_rows[(size_t)b * a.ld_add + row];
  if (a.add_vec) e.vec = a.add_vec[row];
}
__device__ __forceinline__ float residual_out(const GemvBf16& a, int row, int b, const ResidualElem& e, float v) {
  float s = e.old + v;
  if (a.add_rows) s += e.rows;
  if (a.add_vec) s += e.vec;
  a.out[(size_t)b * a.ldo + row] = s;
  return s;
}
template <int OUT>
__device__ __forceinline__ void gemv_out(const GemvBf16& a, int row, int b, float v) {
  float* o = a.out + (size_t)b * a.ldo + row;
  if constexpr (OUT == GEMV_OUT_STORE) *o = v;
  if constexpr (OUT == GEMV_OUT_ACT) *o = act_ranges(a.bias ? v + a.bias[row] : v, row, a.act);
  if constexpr (OUT == GEMV_OUT_XIELU) *o = xielu_apply(v, a.xielu[0], a.xielu[1]);
  if constexpr (OUT == GEMV_OUT_SOFTCAP) *o = soft_cap(v, a.cap);
}

// GEMV_OUT_STREAMS: what the thread that will have (row, b) needs, requested ahead of the products
struct StreamElem {
  float old[HC_MAX], bias = 0.f;
};
__device__ __forceinline__ void stream_elem_load(const GemvBf16& a, int row, int b, StreamElem& e) {
  stream_load(a.sm, a.out + (size_t)b * a.ldo + row, e.old);
  if (a.bias) e.bias = a.bias[row];
}
__device__ __forceinline__ float stream_elem_mix(const GemvBf16& a, int row, int b, const StreamElem& e, float v) {
  return stream_apply(a.sm, a.out + (size_t)b * a.ldo + row, e.old, v + e.bias);
}
__device__ __forceinline__ void stream_elem_out(const GemvBf16& a, int row, int b, const StreamElem& e, float v) {
  a.u[(size_t)b * a.ldo + row] = stream_elem_mix(a, row, b, e, v);
}
// columns of a piece of a row's square sum: a workgroup of the batched linears below owns as many at least
__host__ __device__ inline int ss_columns(int rows) { return rows <= 8 ? 8 : 16; }
// v of 8 or 16 neighbouring columns in as many lanes (zero outside the matrix): what the next linear reads, and its square sum.  Without out16: as f32.
// gain: gain_out[row] (1 without)
__device__ __forceinline__ void rows16_out(const GemvBf16& a, int row, int b, float v, float gain) {
  const bool in = b < a.nb && row < a.N;
  if (!a.out16) {
    if (in) a.u[(size_t)b * a.ldo + row] = v;
    return;
  }
  if (in) a.out16[(size_t)b * a.ldo + row] = f2bf(a.gain_out ? v * gain : v);
  float s = group_sum<8>(v * v);
  if (a.nb <= 8) {  // (ss_columns)
    if (in && (row & 7) == 0) a.ss_out[(size_t)b * a.ld_ss_out + (row >> 3)] = s;
    return;
  }
  s += dpp_f<0x140>(s);
  if (in && (row & 15) == 0) a.ss_out[(size_t)b * a.ld_ss_out + (row >> 4)] = s;
}

#define GEMV_BF16_LDS_FLOATS 8192  // rhs elements staged at a time, all rows together: a cut segment is a multiple of the steps in flight

// WV: waves of a workgroup; UN: steps of 512 in flight; NT: weights nontemporal (GemvBf16::resident); ROLL: a step's registers are refilled as soon as it has been used, else all
// of them are asked for together in front of the products
template <int WV, int NB, int R, int UN, int IN, int OUT, bool NT, bool ROLL>
__global__ __launch_bounds__(64 * WV) void k_gemv_bf16(const GemvBf16 a) {
  extern __shared__ __attribute__((aligned(16))) float gemv_lds[];  // [NB][2][seg / 2]
  __shared__ float red[WV][NB];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg();
  const int row0 = (blockIdx.x * WV + wave) * R, b0 = blockIdx.y * NB;
  const int seg = a.K < GEMV_BF16_LDS_FLOATS / NB ? a.K : GEMV_BF16_LDS_FLOATS / NB;  // elements per staged segment (512-multiple if cut)
  const int half = seg / 2;                                                           // floats per half-octet plane
  const unsigned short* wr[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int row = row0 + r < a.N ? row0 + r : a.N - 1;
    wr[r] = a.w + (size_t)row * a.ldw;
  }
  i32x4 wv[UN][R];
  auto request = [&](int u, int k0) {
    int k = k0 + u * 512 + lane * 8;
    k = k < a.K ? k : 0;  // (a lane past the end requests the row's start and never uses it)
#pragma unroll
    for (int r = 0; r < R; r++) wv[u][r] = ld<NT>((const i32x4*)(wr[r] + k));
  };
#pragma unroll
  for (int u = 0; u < UN; u++) request(u, 0);
  StreamElem elem;  // of lane r NB + b
  const int my_row = row0 + lane / NB, my_b = b0 + lane % NB;
  const bool mine = (OUT == GEMV_OUT_STREAMS || OUT == GEMV_OUT_RESIDUAL) && lane < R * NB && my_row < a.N && my_b < a.nb;
  ResidualElem res;
  if constexpr (OUT == GEMV_OUT_RESIDUAL) residual_load(a, my_row < a.N ? my_row : a.N - 1, my_b < a.nb ? my_b : a.nb - 1, res);  // (no branch on the lane)
  if constexpr (OUT == GEMV_OUT_STREAMS) {
    static_assert(R * NB <= 64, "a lane per result");
    if (mine) stream_elem_load(a, my_row, my_b, elem);
  }
  float acc[R][NB];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[r][b] = 0.f;
  float tail[NB], sq[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    sq[b] = 0.f;
    tail[b] = 1.f;
  }
  if constexpr (IN == GEMV_IN_SPLIT) {
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int bb = b0 + b < a.nb ? b0 + b : a.nb - 1;
      float s = 0.f;
      for (int i = lane; i < a.n_ss; i += 64) s += a.ss[(size_t)bb * a.ld_ss + i];
      s = wave_sum_f32(s);
      tail[b] = 1.0f / sqrtf(s / (float)a.mean_n + a.eps);
    }
  }
  for (int s0 = 0; s0 < a.K; s0 += seg) {
    const int n = a.K - s0 < seg ? a.K - s0 : seg;
    if (s0 > 0) __syncthreads();  // the previous segment has been read by every wave
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int bb = b0 + b < a.nb ? b0 + b : a.nb - 1;
      const float* xr = a.x + (size_t)bb * a.ldx + s0;
      float* lo = gemv_lds + b * 2 * half;
      for (int q = tid; q < n / 8; q += 64 * WV) {
        f32x4 v0 = *(const f32x4*)(xr + q * 8), v1 = *(const f32x4*)(xr + q * 8 + 4);
        if constexpr (IN == GEMV_IN_RMS || IN == GEMV_IN_RMSV) {
#pragma unroll
          for (int e = 0; e < 4; e++) sq[b] = __builtin_fmaf(v0[e], v0[e], __builtin_fmaf(v1[e], v1[e], sq[b]));
        }
        if constexpr (IN == GEMV_IN_RMSV) {
          v0 *= *(const f32x4*)(a.gain + s0 + q * 8);
          v1 *= *(const f32x4*)(a.gain + s0 + q * 8 + 4);
        }
        if constexpr (IN == GEMV_IN_SPLIT) {
          if (s0 + q * 8 >= a.k_split) {
            v0 *= tail[b];
            v1 *= tail[b];
          }
        }
        *(f32x4*)(lo + q * 4) = v0;
        *(f32x4*)(lo + half + q * 4) = v1;
      }
    }
    if constexpr (IN == GEMV_IN_RMS || IN == GEMV_IN_RMSV) {
      if (s0 + seg >= a.K) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
          const float s = wave_sum_f32(sq[b]);
          if (lane == 0) red[wave][b] = s;
        }
      }
    }
    __syncthreads();
    // UN steps; MORE: a step's registers take the one UN steps further.  (A check a step would end the loads in flight.)
    auto steps = [&](auto Mc, int k0, const i32x4 (&w)[UN][R]) {
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int k = k0 + u * 512 + lane * 8;
        if (k < n) {
#pragma unroll
          for (int b = 0; b < NB; b++) {
            const float* lo = gemv_lds + b * 2 * half + (k >> 1);
            const f32x4 x0 = *(const f32x4*)lo, x1 = *(const f32x4*)(lo + half);
#pragma unroll
            for (int r = 0; r < R; r++) {
              float s = acc[r][b];
#pragma unroll
              for (int e = 0; e < 2; e++) {
                const unsigned p = (unsigned)w[u][r][e], p2 = (unsigned)w[u][r][e + 2];
                s = __builtin_fmaf(__builtin_bit_cast(float, p << 16), x0[2 * e], s);
                s = __builtin_fmaf(__builtin_bit_cast(float, p & 0xffff0000u), x0[2 * e + 1], s);
                s = __builtin_fmaf(__builtin_bit_cast(float, p2 << 16), x1[2 * e], s);
                s = __builtin_fmaf(__builtin_bit_cast(float, p2 & 0xffff0000u), x1[2 * e + 1], s);
              }
              acc[r][b] = s;
            }
          }
        }
        if constexpr (decltype(Mc)::value) request(u, s0 + k0 + UN * 512);  // (also across a segment's end: seg % (UN * 512) == 0 then)
      }
    };
    for (int k0 = 0; k0 < n; k0 += UN * 512) {
      const bool more = s0 + k0 + UN * 512 < a.K;
      if constexpr (ROLL) {
        if (more)
          steps(std::true_type{}, k0, wv);
        else
          steps(std::false_type{}, k0, wv);
      } else {
        i32x4 cur[UN][R];
#pragma unroll
        for (int u = 0; u < UN; u++)
#pragma unroll
          for (int r = 0; r < R; r++) cur[u][r] = wv[u][r];
        if (more) {
#pragma unroll
          for (int u = 0; u < UN; u++) request(u, s0 + k0 + UN * 512);
        }
        steps(std::false_type{}, k0, cur);
      }
    }
  }
  float scale[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    scale[b] = 1.f;
    if constexpr (IN == GEMV_IN_RMS || IN == GEMV_IN_RMSV) {
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < WV; w += 4) s += (red[w][b] + red[w + 1][b]) + (red[w + 2][b] + red[w + 3][b]);
      scale[b] = (IN == GEMV_IN_RMS ? *a.gain : 1.0f) / sqrtf(s / (float)a.mean_n + a.eps);
    }
  }
  if constexpr (OUT == GEMV_OUT_GLU) {
    static_assert(R % 2 == 0, "a wave holds both rows of a pair");
#pragma unroll
    for (int r = 0; r < R; r += 2)
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float gate = wave_sum_f32(acc[r][b]) * scale[b], up = wave_sum_f32(acc[r + 1][b]) * scale[b];
        const int row = row0 + r, bb = b0 + b;
        if (lane == ((r / 2 * NB + b) & 63) && row < a.N && bb < a.nb) a.out[(size_t)bb * a.ldo + row / 2] = gelu_tanh(gate) * up;
      }
    return;
  }
  if constexpr (OUT == GEMV_OUT_STREAMS || OUT == GEMV_OUT_RESIDUAL) {
    float y = 0.f;
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float v = wave_sum_f32(acc[r][b]) * scale[b];
        y = lane == r * NB + b ? v : y;
      }
    if constexpr (OUT == GEMV_OUT_STREAMS) {
      if (mine) stream_elem_out(a, my_row, my_b, elem, y);
    } else {
      if (mine) (void)residual_out(a, my_row, my_b, res, y);
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const float v = wave_sum_f32(acc[r][b]) * scale[b];
      const int row = row0 + r, bb = b0 + b;
      if (lane == ((r * NB + b) & 63) && row < a.N && bb < a.nb) {
        gemv_out<OUT>(a, row, bb, v);
      }
    }
}

// ---- the same linear for 3 .. 16 rhs rows: one pass over the weights on the matrix cores ---------------------------------------------
// A workgroup of W waves owns 16 RT weight rows; the waves take the 64-element pieces of k in turn, D pieces of requests out each, and their
// tiles are added through LDS at the end.  The rhs becomes bf16 on the way: rounded (SPL = 1), or as three exact pieces (SPL = 3; see
// split_store in gemm_bf16.hpp) -- or arrives as bf16 (GEMV_IN_BF16).  K is a multiple of 64.
//
// A fragment of the matrix instruction has a row per lane, so neighbouring lanes' 16 bytes would come from different cache lines: 64 line
// accesses per request, and that -- not the bytes -- was the bound (2048 x 8192, 16 rows: 23.2 us, 20 of them 128 pieces x 6 requests x
// 64 accesses of one CU).  Here eight (f32 rhs: sixteen) neighbouring lanes take a row's 128 (256) bytes and the tile goes through the
// wave's own 2 KB of LDS, 16-byte pieces permuted by (row / 2) % 8 as in gemm_bf16.hip; no barrier, a wave's LDS accesses are in order.
// 16 rows, before -> after, with bf16 rows: 2048 x 8192 23.2 -> 12.7 us, 2048 x 4096 17.5 -> 8.6, 5632 x 2048 19.3 -> 13.9, 8192 x 2048
// 14.1 -> 10.2, 32000 x 2048 35.4 -> 30.3 (4.3 TB/s); what is left is a launch's ramp, two rounds of memory latency and the hand-over.
// NTW: weights past the caches' replacement, so that the 16 rows of the rhs, which every workgroup reads whole, stay (GemvBf16::resident).  16 x 154
// tokens of 4 layers of width 2048 20054 -> 18687 us, 4 x 716 of latent and windowed layers 7443 -> 7283.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
// f32 -> its upper, middle and lower eight significand bits as bf16: their sum is exact
__device__ __forceinline__ void split3(float v, unsigned short& hi, unsigned short& mid, unsigned short& lo) {
  const float a = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) & 0xffff0000u), r = v - a;
  const float b = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, r) & 0xffff0000u);
  hi = (unsigned short)(__builtin_bit_cast(unsigned, a) >> 16);
  mid = (unsigned short)(__builtin_bit_cast(unsigned, b) >> 16);
  lo = f2bf(r - b);
}
__device__ __forceinline__ void split3(const float (&v)[8], bf16x8& hi, bf16x8& mid, bf16x8& lo) {
  unsigned short h[8], m[8], l[8];
#pragma unroll
  for (int e = 0; e < 8; e++) split3(v[e], h[e], m[e], l[e]);
  __builtin_memcpy(&hi, h, 16);
  __builtin_memcpy(&mid, m, 16);
  __builtin_memcpy(&lo, l, 16);
}
// what this wave has written to LDS is there for its other lanes (a wave's LDS accesses are in order; the compiler is told)
__device__ __forceinline__ void wave_lds_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }
__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// XG: f32 rows are requested and split in groups of four, as many as there are rows -- a group is a request, twelve conversions and three LDS
// stores a lane and piece, which three rows of four groups paid for in full (f32 compute, us, 4 rows, all groups / one: 11264 x 2048
// 17.3 / 12.2, gate | up of 16384 x 2048 18.5 / 16.1).
// XG = 1 and bf16 rows: up to eight of them, one request for a piece instead of two.
// HALF (up to eight rows): a workgroup owns 8 weight rows, where 16 would leave half of the CUs without one (a CU draws some 25 KB/us, however much it asks
// for).  A step is the next two pieces of k that the wave would take of 16 rows, their eight weight rows one above the other in the tile, and each is
// multiplied by its piece of the rhs in turn (the lower and the upper half of the product are the same).  Us a launch, 4
// rows, streams behind it: 2048 x 8192 11.3 -> 8.5, 2048 x 2048 with a tail 6.3 -> 5.4.  (16 rows, whose rhs is as many bytes as the weights of 16 rows: 2048 x
// 8192 12.2 -> 11.7, 2048 x 4096 6.2 -> 6.8; twice as many pieces of square sums to read cost the linears behind them more.)
// KS = 2 (nine rows and more, the same matrices from GEMV16_SHARED_K columns on): two workgroups of eight waves share a tile's k, each with the pieces that eight of the sixteen
// waves would take, and meet at the end (below): 16 rows, residual behind it, 2048 x 8192 12.0 -> 9.0 us, 2048 x 4096 7.4 -> 6.4, 1280 x 4096 7.1 -> 6.0; 2048 x 2048 5.0 -> 5.1.
// The sums of bf16 rows are the same in every form: pieces of k by wave, waves in order (from GEMV16_SHARED_K columns on those of narrow matrices in two halves), square
// sums of 16 columns: a sequence's logits do not depend on how many others, three to sixteen rows in all, share its step.
#define GEMV16_SHARED_K 3072
template <int RT, int SPL, int W, int D, int IN, int OUT, bool NTW, int XG = 4, bool HALF = false, int KS = 1>
__global__ __launch_bounds__(64 * W) void k_gemv16_bf16(const GemvBf16 a) {
  constexpr int LD = 20, NT = 64 * W;
  constexpr bool XB = IN == GEMV_IN_BF16 || IN == GEMV_IN_BF16_RMS || IN == GEMV_IN_BF16_SPLIT, NORM = IN == GEMV_IN_RMS || IN == GEMV_IN_RMSV;
  constexpr bool PIECES = IN == GEMV_IN_BF16_RMS || IN == GEMV_IN_BF16_SPLIT, TAIL = IN == GEMV_IN_BF16_SPLIT;
  constexpr int XR = XB ? (XG == 1 ? 1 : 2) : XG;  // requests for a piece of the rhs
  constexpr int WR = HALF ? 8 : 16 * RT, KP = HALF ? 2 : 1;  // weight rows of the workgroup; pieces of k a step
  static_assert(!XB || SPL == 1, "a bf16 rhs has one piece");
  constexpr bool EIGHT = XB && XG == 1;
  static_assert(!HALF || (EIGHT && RT == 1), "eight weight rows: up to eight bf16 rows");
  union Lds {
    unsigned short in[W][RT + SPL * KP][16 * 64];  // a wave's tiles: weights, rhs
    float tile[W][RT][16 * LD];
  };
  __shared__ __attribute__((aligned(16))) Lds lds;
  __shared__ float sums[W][16], scale[16];
  static_assert(KS == 1 || (KS == 2 && RT == 1 && !HALF && XB && W >= 4), "two workgroups a tile: one of 16 weight rows, bf16 rows");
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg(), fr = lane & 15, fk = lane >> 4;
  // (KS = 2: the two of a tile are eight workgroups apart, on one XCD: what was touched there for the tile's rows serves both)
  const int tile = KS == 2 ? (blockIdx.x >> 4) * 8 + (blockIdx.x & 7) : blockIdx.x, part = KS == 2 ? (blockIdx.x >> 3) & 1 : 0;
  if (KS == 2 && tile * WR >= a.N) return;
  const int row0 = tile * WR, kw = part * W + wave;  // kw: this wave's place among those of k
  // where this lane's part of a request lies: 16 bytes, eight lanes a row (f32: sixteen)
  const int r8 = lane >> 3, c8 = lane & 7, r16 = lane >> 4, c16 = lane & 15;
  // (32-bit offsets from a scalar base)
  const char *wb = (const char*)(a.w + (size_t)row0 * a.ldw), *xbase = XB ? (const char*)a.x16 : (const char*)a.x, *gb = (const char*)a.gain;
  unsigned wo[RT][2], xo[XR];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int row = HALF ? r8 : t * 16 + j * 8 + r8;
      wo[t][j] = (unsigned)(row0 + row < a.N ? row : a.N - 1 - row0) * (unsigned)a.ldw * 2 + c8 * 16;
    }
#pragma unroll
  for (int j = 0; j < XR; j++) {
    const int b = XB ? j * 8 + r8 : j * 4 + r16;
    xo[j] = (unsigned)(b < a.nb ? b : a.nb - 1) * (unsigned)a.ldx * (XB ? 2 : 4) + (XB ? c8 : c16) * 16;
  }
  i32x4 wv[D][RT][2], xv[D][KP * XR];
  f32x4 gv[D];
  const int n = a.K / 64, last = n - 1;
  constexpr int S = KP * W * KS;  // pieces from a step of this wave's to its next
  auto request = [&](int d, int i) {
    const char *w = wb + i * 128, *x = xbase + i * (XB ? 128 : 256);
    const int second = HALF && i + W < n ? 128 * W : 0;  // (none: itself again, not used)
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int j = 0; j < 2; j++) wv[d][t][j] = ld<NTW>((const i32x4*)(w + (HALF ? j * second : 0) + wo[t][j]));
#pragma unroll
    for (int h = 0; h < KP; h++)
#pragma unroll
      for (int j = 0; j < XR; j++) xv[d][h * XR + j] = *(const i32x4*)(x + h * second + xo[j]);
    if constexpr (IN == GEMV_IN_RMSV) gv[d] = *(const f32x4*)(gb + i * 256 + (unsigned)c16 * 16);
  };
  // A row's sum of squares, by pieces of 16 columns (two of 8): piece q + QT u belongs to term q, in the order of u, the terms meet by neighbours, pairs, ...  As many
  // terms as four a wave of all that share k, so that two workgroups of eight waves have sixteen waves' sum.  A lane
  // requests 16 bytes -- QC neighbouring terms of one u, QU of which a row's QR threads have at a time -- the first ahead of the weights (loads come back in order).
  constexpr bool QTWO = EIGHT && !TAIL;
  constexpr int QT = 4 * W * KS, QC = QTWO ? 2 : 4, QL = QT / QC, QR = QTWO ? 64 : NT / 16, QU = QR / QL;
  const int q_row = tid / QR, q_at = tid % QR, q_j = q_at % QL, q_u = q_at / QL, n4 = (a.n_ss + 3) / 4;
  const f32x4* q_ss = PIECES ? (const f32x4*)(a.ss + (size_t)(q_row < a.nb ? q_row : a.nb - 1) * a.ld_ss) : nullptr;
  f32x4 q_v = {0.f, 0.f, 0.f, 0.f};
  if constexpr (PIECES) q_v = q_ss[q_u * QL + q_j < n4 ? q_u * QL + q_j : 0];
  float tail[XR], sq[XR];  // of row 4 j + r16
  const float* t_ss[XR];
#pragma unroll
  for (int j = 0; j < XR; j++) {
    tail[j] = sq[j] = 0.f;
    if constexpr (IN == GEMV_IN_SPLIT) {  // (the first pieces of every row: ahead of the weights, too)
      t_ss[j] = a.ss + (size_t)(j * 4 + r16 < a.nb ? j * 4 + r16 : a.nb - 1) * a.ld_ss;
      tail[j] = t_ss[j][c16 < a.n_ss ? c16 : 0];
    }
  }
  unsigned launch = 0;
  if constexpr (KS == 2) launch = __hip_atomic_load(a.meet + tile * 4 + (wave & 3), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (kw < n) {
#pragma unroll
    for (int d = 0; d < D; d++) request(d, kw + d * S < n ? kw + d * S : last);  // (clamped: no branch between the requests)
  }
  float out_c[2] = {0.f, 0.f};  // (asked for here: behind the products they would be one more round trip of every workgroup)
  if constexpr (OUT == GEMV_OUT_XIELU) {
    out_c[0] = a.xielu[0];
    out_c[1] = a.xielu[1];
  }
  const float gain1 = PIECES && !TAIL && a.gain ? *a.gain : 1.0f;
  constexpr int RB = HALF ? 3 : 4, ELEMS = (WR * 16 + NT - 1) / NT;
  // result j of the tile: weight row t 16 + r of the workgroup, row b of the rhs
  auto of = [&](int j, int& t, int& b, int& r) {
    t = j >> 8;
    b = (j >> RB) & 15;
    r = j & ((1 << RB) - 1);
  };
  StreamElem elem[ELEMS];  // of this thread's results: element tid + NT i of the tile
  ResidualElem res[ELEMS];
  float gain_next[ELEMS];
  if constexpr (OUT == GEMV_OUT_RESIDUAL || OUT == GEMV_OUT_STREAMS) {
#pragma unroll
    for (int i = 0; i < ELEMS; i++) {
      int t, b, r;
      of(tid + i * NT < WR * 16 ? tid + i * NT : 0, t, b, r);
      const int row = row0 + t * 16 + r < a.N ? row0 + t * 16 + r : a.N - 1;
      gain_next[i] = a.gain_out ? a.gain_out[row] : 1.f;
      if constexpr (OUT == GEMV_OUT_RESIDUAL) residual_load(a, row, b < a.nb ? b : a.nb - 1, res[i]);
    }
  }
  if constexpr (OUT == GEMV_OUT_STREAMS) {
#pragma unroll
    for (int i = 0; i < ELEMS; i++) {
      const int j = tid + i * NT;
      int t, b, r;
      of(j, t, b, r);
      const int row = row0 + t * 16 + r;
      if (j < WR * 16 && b < a.nb && row < a.N) stream_elem_load(a, row, b, elem[i]);
    }
  }
  if constexpr (IN == GEMV_IN_SPLIT) {
#pragma unroll
    for (int j = 0; j < XR; j++) {
      float t = c16 < a.n_ss ? tail[j] : 0.f;
      for (int i = c16 + 16; i < a.n_ss; i += 16) t += t_ss[j][i];
      tail[j] = 1.0f / sqrtf(row16_sum_f32(t) / (float)a.mean_n + a.eps);
    }
  }
  f32x4 acc[RT], acc2[RT];  // (TAIL: what is normalized apart)
#pragma unroll
  for (int t = 0; t < RT; t++) acc[t] = acc2[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned short(*mine)[16 * 64] = lds.in[wave];
  auto multiply = [&](const i32x4 (&wc)[RT][2], const i32x4 (&xc)[KP * XR], const f32x4& gc, int i) {
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int r = j * 8 + r8;
        *(i32x4*)&mine[t][r * 64 + ((c8 ^ ((r >> 1) & 7)) * 8)] = wc[t][j];
      }
    if constexpr (XB) {
#pragma unroll
      for (int h = 0; h < KP; h++)
#pragma unroll
        for (int j = 0; j < XR; j++) {  // (rows 8 .. 15 that are not there: whatever LDS holds, in columns that are not stored)
          const int r = j * 8 + r8;
          *(i32x4*)&mine[RT + h][r * 64 + ((c8 ^ ((r >> 1) & 7)) * 8)] = xc[h * XR + j];
        }
    } else {
#pragma unroll
      for (int j = 0; j < XR; j++) {
        const int r = j * 4 + r16;
        f32x4 v = __builtin_bit_cast(f32x4, xc[j]);
        if constexpr (NORM) {
#pragma unroll
          for (int e = 0; e < 4; e++) sq[j] = __builtin_fmaf(v[e], v[e], sq[j]);
        }
        if constexpr (IN == GEMV_IN_RMSV) v *= gc;
        if constexpr (IN == GEMV_IN_SPLIT) v *= i * 64 >= a.k_split ? tail[j] : 1.f;  // (k_split is a multiple of 64)
        unsigned short p[SPL][4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if constexpr (SPL == 1)
            p[0][e] = f2bf(v[e]);
          else
            split3(v[e], p[0][e], p[1][e], p[2][e]);
        }
#pragma unroll
        for (int q = 0; q < SPL; q++) {
          i32x2 w;
          __builtin_memcpy(&w, p[q], 8);
          *(i32x2*)&mine[RT + q][r * 64 + (((c16 >> 1) ^ ((r >> 1) & 7)) * 8) + (c16 & 1) * 4] = w;
        }
      }
    }
    wave_lds_order();
    if constexpr (HALF) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int at = i + h * W;
        if (at >= n) break;  // (uniform)
        const bool apart = TAIL && at * 64 >= a.k_split;
        const int r = h * 8 + (fr & 7);
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const bf16x8 w = *(const bf16x8*)&mine[0][r * 64 + (((u * 4 + fk) ^ ((r >> 1) & 7)) * 8)];
          const bf16x8 x = *(const bf16x8*)&mine[1 + h][fr * 64 + (((u * 4 + fk) ^ ((fr >> 1) & 7)) * 8)];
          if (apart)
            acc2[0] = mfma_bf16(w, x, acc2[0]);
          else
            acc[0] = mfma_bf16(w, x, acc[0]);
        }
      }
      wave_lds_order();
      return;
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int at = fr * 64 + (((u * 4 + fk) ^ ((fr >> 1) & 7)) * 8);
      bf16x8 x[SPL];
#pragma unroll
      for (int q = 0; q < SPL; q++) x[q] = *(const bf16x8*)&mine[RT + q][at];
#pragma unroll
      for (int t = 0; t < RT; t++) {
        const bf16x8 w = *(const bf16x8*)&mine[t][at];
        if (TAIL && i * 64 >= a.k_split)
          acc2[t] = mfma_bf16(w, x[0], acc2[t]);
        else
#pragma unroll
          for (int q = SPL - 1; q >= 0; q--) acc[t] = mfma_bf16(w, x[q], acc[t]);  // (the smallest piece first)
      }
    }
    wave_lds_order();
  };
  for (int i = kw; i < n; i += D * S) {
    if (i + D * S < n) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        multiply(wv[d], xv[d], gv[d], i + d * S);
        request(d, i + (D + d) * S < n ? i + (D + d) * S : last);
      }
    } else {
#pragma unroll
      for (int d = 0; d < D; d++)
        if (i + d * S < n) multiply(wv[d], xv[d], gv[d], i + d * S);
    }
  }
  if constexpr (NORM) {
#pragma unroll
    for (int j = 0; j < XR; j++) {
      const float t = row16_sum_f32(sq[j]);
      if (c16 == 0) sums[wave][j * 4 + r16] = t;
    }
  }
  if constexpr (PIECES) {
    float term[QC] = {};
    for (int u0 = 0; u0 * QL < n4; u0 += QU) {
      const int at = (u0 + q_u) * QL + q_j;
      if (u0 > 0) q_v = q_ss[at < n4 ? at : 0];
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = 4 * at + e < a.n_ss ? q_v[e] : 0.f;  // (behind the last piece: whatever is there)
      float p[QC];
#pragma unroll
      for (int c = 0; c < QC; c++) p[c] = QTWO ? v[2 * c] + v[2 * c + 1] : v[c];
#pragma unroll
      for (int s = 0; s < QU; s++) {
        if ((u0 + s) * QL >= n4) break;  // (uniform)
#pragma unroll
        for (int c = 0; c < QC; c++) term[c] += s == 0 ? p[c] : __shfl(p[c], (lane & ~(QR - 1)) + s * QL + q_j, 64);  // (what is used is in the lanes of u = 0)
      }
    }
    float t = QC == 2 ? term[0] + term[1] : (term[0] + term[1]) + (term[QC - 2] + term[QC - 1]);
    t = group_sum<8>(t);
    if constexpr (QL >= 16) t += dpp_f<0x140>(t);
    if constexpr (QL == 32) t += __shfl_xor(t, 16, 64);
    if (q_at == 0 && q_row < 16) scale[q_row] = gain1 / sqrtf(t / (float)a.mean_n + a.eps);
  }
  __syncthreads();  // (the tiles of results take the place of the operands')
  if constexpr (TAIL) {
#pragma unroll
    for (int t = 0; t < RT; t++) acc[t] += acc2[t] * scale[fr];
  }
  // lane: weight rows 4 fk .. of rhs row fr
#pragma unroll
  for (int t = 0; t < RT; t++) *(f32x4*)&lds.tile[wave][t][fr * LD + fk * 4] = acc[t];
  __syncthreads();
  if constexpr (NORM) {
    if (tid < 16) {
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < W; w++) s += sums[w][tid];
      scale[tid] = (IN == GEMV_IN_RMS ? *a.gain : 1.0f) / sqrtf(s / (float)a.mean_n + a.eps);
    }
    __syncthreads();
  }
  auto met = [&](int t, int b, int r) {  // the waves' sums
    float v = 0.f;
    if constexpr (HALF) {
      float v2 = 0.f;
#pragma unroll
      for (int w = 0; w < W / 2; w++) v += lds.tile[w][t][b * LD + r];
      if (a.K < GEMV16_SHARED_K) v2 = v;
#pragma unroll
      for (int w = W / 2; w < W; w++) v2 += lds.tile[w][t][b * LD + r];
      return a.K < GEMV16_SHARED_K ? v2 : v + v2;
    }
#pragma unroll
    for (int w = 0; w < W; w++) v += lds.tile[w][t][b * LD + r];
    return v;
  };
  float both = 0.f;
  if constexpr (KS == 2) {
    // A wave's 64 results leave as {value, launch} granules before it counts itself in; of the two workgroups' waves the later one takes the other's,
    // which are on their way or there -- it waits for stores that have been issued, never for a workgroup -- and goes on alone.
    if (wave >= 4) return;
    int t, b, r;
    of(tid, t, b, r);
    const float v = met(t, b, r);
    const unsigned tag = (launch >> 1) + 1u;  // (two arrivals a launch: both workgroups see the same half, whether the other one has come or not)
    unsigned long long* g = a.half + (size_t)tile * 512 + tid;
    __hip_atomic_store(g + part * 256, ((unsigned long long)tag << 32) | __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned n_before = 0;
    if (lane == 0) n_before = __hip_atomic_fetch_add(a.meet + tile * 4 + wave, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((__builtin_amdgcn_readfirstlane(n_before) & 1u) == 0) return;
    unsigned long long o;
    do {
      o = __hip_atomic_load(g + (part ^ 1) * 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } while ((unsigned)(o >> 32) != tag);
    const float ov = __builtin_bit_cast(float, (unsigned)o);
    both = v + ov;  // (the same whichever is later)
  }
  if constexpr (OUT == GEMV_OUT_GLU && KS == 2) {
    int t, b, r;
    of(tid, t, b, r);
    const int row = row0 + r;
    float up = dpp_f<0xB1>(both), gate = both;  // (of the neighbour)
    if constexpr (IN == GEMV_IN_BF16_RMS) {
      gate *= scale[b];
      up *= scale[b];
    }
    if ((r & 1) == 0 && b < a.nb && row < a.N) {
      const size_t o = (size_t)b * a.ldo + row / 2;
      if (a.out16)
        a.out16[o] = f2bf(gelu_tanh(gate) * up);
      else
        a.out[o] = gelu_tanh(gate) * up;
    }
    return;
  }
  if constexpr (OUT == GEMV_OUT_GLU) {
    for (int i = tid; i < WR * 8; i += NT) {
      int t, b, r;
      of(2 * i, t, b, r);
      const int row = row0 + t * 16 + r;
      float gate = met(t, b, r), up = met(t, b, r + 1);
      if constexpr (NORM || IN == GEMV_IN_BF16_RMS) {
        gate *= scale[b];
        up *= scale[b];
      }
      if (b < a.nb && row < a.N) {
        const size_t o = (size_t)b * a.ldo + row / 2;
        if (a.out16)
          a.out16[o] = f2bf(gelu_tanh(gate) * up);
        else
          a.out[o] = gelu_tanh(gate) * up;
      }
    }
    return;
  }
  if constexpr (OUT == GEMV_OUT_STREAMS) {
#pragma unroll
    for (int i = 0; i < ELEMS; i++) {
      const int j = tid + i * NT;
      if (j >= WR * 16) break;  // (whole waves)
      int t, b, r;
      of(j, t, b, r);
      const int row = row0 + t * 16 + r;
      float u = 0.f;
      if (b < a.nb && row < a.N) u = stream_elem_mix(a, row, b, elem[i], KS == 2 ? both : met(t, b, r));
      rows16_out(a, row, b, u, gain_next[i]);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < ELEMS; i++) {
    const int j = tid + i * NT;
    if (j >= WR * 16) break;  // (whole waves)
    int t, b, r;
    of(j, t, b, r);
    const int row = row0 + t * 16 + r;
    float v = KS == 2 ? both : met(t, b, r);
    if constexpr (NORM || IN == GEMV_IN_BF16_RMS) v *= scale[b];
    if constexpr (OUT == GEMV_OUT_RESIDUAL) {
      float x = 0.f;
      if (b < a.nb && row < a.N) x = residual_out(a, row, b, res[i], v);
      if (a.out16) rows16_out(a, row, b, x, gain_next[i]);
      continue;
    }
    if (b < a.nb && row < a.N) {
      if constexpr (OUT == GEMV_OUT_XIELU) {
        const float y = xielu_apply(v, out_c[0], out_c[1]);
        if (a.out16)
          a.out16[(size_t)b * a.ldo + row] = f2bf(y);
        else
          a.out[(size_t)b * a.ldo + row] = y;
        continue;
      }
      gemv_out<OUT>(a, row, b, v);
    }
  }
}

// f32 rows, and linears of bf16 rows into the residual: 32 rows a workgroup where that still fills the chip, else 16; sixteen waves where 16 rows leave CUs without
// a workgroup and k is long enough for each of them to have a few steps.  One piece of the rhs: bf16 rows, but for a classifier behind a prompt pass.
// Three pieces of more than eight f32 rows: two steps of requests hold 140 registers a thread, one workgroup a CU; where there are more workgroups than
// CUs, two of them with one step out each are faster (us, 12 rows: 11264 x 2048 18.0 -> 16.4, 8192 x 1024 8.7 -> 6.9), elsewhere they are
// not (2048 x 8192, 128 workgroups: 16.2 -> 19.8).
template <int RT, int SPL, int W, int IN, int OUT, bool NTW, int D0 = 0>
inline void launch_gemv16_t(hipStream_t st, crabml_hip_device::ProfRec* rec, const GemvBf16& a, int n_cu) {
  constexpr int D = D0 ? D0 : IN < GEMV_IN_BF16 || RT == 2 ? 2 : OUT == GEMV_OUT_STREAMS ? 3 : 4;  // (registers: sixteen waves a CU)
  const dim3 grid((a.N + 16 * RT - 1) / (16 * RT));
  if constexpr (IN >= GEMV_IN_BF16) {
    if (a.nb <= 8) {
      launch_k(st, rec, k_gemv16_bf16<RT, SPL, W, D, IN, OUT, NTW, 1>, grid, dim3(64 * W), 0, a);
      return;
    }
  }
  if constexpr (SPL == 3) {
    if (a.nb <= 4) {
      launch_k(st, rec, k_gemv16_bf16<RT, SPL, W, D, IN, OUT, NTW, 1>, grid, dim3(64 * W), 0, a);
      return;
    }
    if (a.nb <= 8) {
      launch_k(st, rec, k_gemv16_bf16<RT, SPL, W, D, IN, OUT, NTW, 2>, grid, dim3(64 * W), 0, a);
      return;
    }
    if (RT == 1 && (int)grid.x > n_cu) {
      launch_k(st, rec, k_gemv16_bf16<RT, SPL, W, 1, IN, OUT, NTW>, grid, dim3(64 * W), 0, a);
      return;
    }
  }
  launch_k(st, rec, k_gemv16_bf16<RT, SPL, W, D, IN, OUT, NTW>, grid, dim3(64 * W), 0, a);
}
// bf16: of the rhs
inline bool gemv16_deep(int N, int K, int n_cu) { return (N + 15) / 16 < n_cu && K >= 2048; }
inline bool gemv16_narrow(int N, int K, int n_cu) { return gemv16_deep(N, K, n_cu) && (N + 15) / 16 * 2 <= n_cu; }
inline int gemv16_rows(bool bf16, int N, int K, int nb, int n_cu) {
  if (N >= 16384) return 32;
  return bf16 && nb <= 8 && gemv16_narrow(N, K, n_cu) ? 8 : 16;
}
// what k shared by two workgroups needs (GemvBf16::half, meet)
inline size_t gemv16_half_bytes(int n_cu) { return (size_t)(n_cu / 2) * 512 * sizeof(unsigned long long); }
inline size_t gemv16_meet_bytes(int n_cu) { return (size_t)(n_cu / 2) * 4 * sizeof(unsigned); }
// More rows of weights than 16 a CU, bf16 rows with a norm: as many tiles of 16 a workgroup as make one round of workgroups.  The rhs comes through the L2s once a
// workgroup, as many bytes as 16 rows of weights, and a second round that leaves most CUs without work costs as much as the first.  Us a launch of 16 / 4 rows,
// workgroups of 16 rows / these: 4608 x 512 5.5 / 4.2 and 4.9 / 3.9, 11264 x 512 7.7 / 4.9 and 6.9 / 4.7, 8192 x 1024 6.95 / 5.6 and 6.1 / 5.4, 12288 x 1024 9.4 / 6.8 and
// 8.25 / 6.5, 4608 x 2048 8.4 / 7.2 and 6.7 / 6.4, 8192 x 2048 9.2 / 8.65 and 7.8 / 7.8, 9216 x 2048 11.4 / 9.6 and 9.65 / 9.1, 11264 x 2048 12.1 / 10.4 and 10.3 / 10.3,
// 14336 x 2048 14.8 / 13.3 and 12.8 / 12.9.  Three tiles: sixteen waves where each has two pieces of k, else eight that start sooner
// (9216 x 1024 6.35 / 6.2).  Two tiles: eight waves with a step each out (16 / 3 rows, workgroups of 16 rows / sixteen waves / these: 4112 x 128 3.26 3.47 3.28 and 3.06 3.31 3.11,
// 8192 x 512 5.9 4.5 4.3 and 5.3 4.3 4.1, 4112 x 1280 6.9 7.2 5.8 and 5.8 6.5 5.3, 8192 x 1536 8.2 8.0 6.9 and 6.8 7.2 6.7, 8192 x 3072 13.6 12.2 10.8 and 11.2 11.4 10.4), but
// sixteen with two where rows are 4 KB, which begin on the same memory channels (4608 x 2048 8.45 7.3 7.4 and 6.75 6.5 6.9, 8192 x 2048 9.4 8.8 9.4 and 7.9 7.9 9.1).
// More than four tiles a CU: workgroups of 48 rows (against 32 rows, two steps out: 32000 x 512 11.2 / 9.1, x 1024 14.5 / 13.5, x 2048 24.9 / 24.0, x 4096 48.5 / 44.0) -- or
// of 32 with a step out, where 48 leave CUs with one workgroup of the two that fit (16400 rows; 16 rows, 32 rows and two steps / 48 / these: x 512 7.4 6.4 5.75, x 1280 11.6
// 11.7 10.6, x 3072 21.4 22.9 21.2) or go on in a second round over long rows (32000 x 2560 32.5 30.1 29.8, x 3072 33.6 34.2 33.3, 65536 x 5120 110 111 110, 3 rows 28.3 27.6 26.4,
// 30.6 32.0 31.0, 97 102 98; x 2048 25.2 24.5 24.0, 65536 x 2048 48.1 45.4 46.7 with 3 rows; one full round: 20000 x 2560 24.3 21.1 22.3).  Never with rows of 8 KB (32000 x
// 4096 49.8 44.4 48.7).
// From 4096 columns on eight rows and fewer are as fast or faster in workgroups of 16 (8192 x 4096 12.6 / 15.2).
template <int SPL, int IN, int OUT, bool NTW>
inline bool launch_gemv16_round(hipStream_t st, crabml_hip_device::ProfRec* rec, const GemvBf16& a, int n_cu) {
  const int tiles = (a.N + 15) / 16, per = (tiles + n_cu - 1) / n_cu;
  if (per > 4) {
    const int wgs = (a.N + 47) / 48;
    if (a.K % 4096 != 0 && (2 * wgs < 3 * n_cu || (a.K > 2048 && wgs > 2 * n_cu)))
      launch_gemv16_t<2, SPL, 8, IN, OUT, NTW, 1>(st, rec, a, n_cu);
    else
      launch_gemv16_t<3, SPL, 8, IN, OUT, NTW, 1>(st, rec, a, n_cu);
    return true;
  }
  if (per < 2 || a.K >= 4096) return false;
  if (per == 2 && a.K % 2048 != 0)
    launch_gemv16_t<2, SPL, 8, IN, OUT, NTW, 1>(st, rec, a, n_cu);
  else if (per == 2)
    launch_gemv16_t<2, SPL, 16, IN, OUT, NTW, 2>(st, rec, a, n_cu);
  else if (per == 3 && a.K <= 1024)
    launch_gemv16_t<3, SPL, 8, IN, OUT, NTW, 1>(st, rec, a, n_cu);
  else if (per == 3)
    launch_gemv16_t<3, SPL, 16, IN, OUT, NTW, 1>(st, rec, a, n_cu);
  else
    launch_gemv16_t<4, SPL, 8, IN, OUT, NTW, 1>(st, rec, a, n_cu);
  return true;
}
template <int SPL, int IN, int OUT, bool NTW>
inline void launch_gemv16_n(hipStream_t st, crabml_hip_device::ProfRec* rec, const GemvBf16& a, int n_cu) {
  if constexpr (IN == GEMV_IN_BF16_RMS) {
    if (launch_gemv16_round<SPL, IN, OUT, NTW>(st, rec, a, n_cu)) return;
  }
  const int rows = gemv16_rows(IN >= GEMV_IN_BF16, a.N, a.K, a.nb, n_cu);
  if (rows == 32) {
    launch_gemv16_t<2, SPL, 8, IN, OUT, NTW>(st, rec, a, n_cu);
    return;
  }
  if constexpr (IN >= GEMV_IN_BF16) {
    if (rows == 8) {
      // (two steps out a wave: three or four, of neighbouring pieces of k, made a whole decode step of 3 to 8 rows 0.5 to 3 % longer)
      launch_k(st, rec, k_gemv16_bf16<1, SPL, 16, 2, IN, OUT, NTW, 1, true>, dim3((a.N + 7) / 8), dim3(1024), 0, a);
      return;
    }
    if (gemv16_narrow(a.N, a.K, n_cu) && a.K >= GEMV16_SHARED_K) {
      launch_k(st, rec, k_gemv16_bf16<1, SPL, 8, 2, IN, OUT, NTW, 4, false, 2>, dim3((a.N + 127) / 128 * 16), dim3(512), 0, a);
      return;
    }
    if (gemv16_deep(a.N, a.K, n_cu)) {
      launch_gemv16_t<1, SPL, 16, IN, OUT, NTW>(st, rec, a, n_cu);
      return;
    }
  }
  launch_gemv16_t<1, SPL, 8, IN, OUT, NTW>(st, rec, a, n_cu);
}
template <int SPL, int IN, int OUT>
inline void launch_gemv16_bf16(hipStream_t st, crabml_hip_device::ProfRec* rec, const GemvBf16& a, int n_cu) {
  a.resident ? launch_gemv16_n<SPL, IN, OUT, false>(st, rec, a, n_cu) : launch_gemv16_n<SPL, IN, OUT, true>(st, rec, a, n_cu);
}

template <int WV, int NB, int R, int UN, int IN, int OUT, bool ROLL = true>
inline void launch_gemv_bf16_t(hipStream_t st, crabml_hip_device::ProfRec* rec, const GemvBf16& a) {
  const int cap = GEMV_BF16_LDS_FLOATS / NB, seg = a.K < cap ? a.K : cap;
  launch_k(st, rec, a.resident ? k_gemv_bf16<WV, NB, R, UN, IN, OUT, false, ROLL> : k_gemv_bf16<WV, NB, R, UN, IN, OUT, true, ROLL>,
           dim3((a.N + WV * R - 1) / (WV * R), (a.nb + NB - 1) / NB), dim3(64 * WV), (size_t)NB * seg * sizeof(float), a);
}
// One row of the rhs: every workgroup stages it for itself, so eight waves with a row each are faster than four with one, two or four (half as many copies of the rhs
// through the L2s and half as many workgroups to start, as many requests out from the beginning); a wave has no more requests out than its row has steps -- more are the row's
// start again, 0.1 to 0.2 us each -- and eight where there are more than eight to make, if the rows are at most 2048 or long enough for a round with less than eight to make
// to be a small part (four / eight steps out: 2048 x 5120 6.6 / 6.4, 8192 x 5120 14.9 / 15.5, 16384 x 5120 26.6 / 27.2, 3072 x 8192 10.6 / 10.3, 8192 x 8192 22.7 / 22.6).  What else: two rows a wave where there are more than 8192 of less than 2048
// columns (four of at most 512), four waves up to 1024 rows of longer ones and, but for an rhs that is staged with a gain per element (GEMV_IN_RMSV: twice the bytes a
// workgroup), from 16384 rows of 2048 columns on.  Us a launch, four waves of as many rows as
// was best for them and four or eight steps out / these: 2048 x 512 3.25 / 2.8, 32000 x 512 9.7 / 7.5, 32000 x 128 8.5 / 5.2, 4096 x 1024 4.4 / 4.0, 3648 x 2048 5.5 / 5.0,
// 8192 x 2048 7.7 / 7.4, 11264 x 2048 9.7 / 9.3, 2048 x 8192 7.75 / 7.5, 2048 x 4096 5.2 / 5.1; gate | up of 16384 x 2048 13.7 / 12.7, 8192 x 512 4.6 / 4.1.
// A row a wave from 16384 rows on, four waves / eight: with one gain 32000 x 2048 20.7 / 20.7, x 4096 38.8 / 40.5, 128256 x 4096 146 / 153; with a gain per element 16384 x
// 2048 14.0 / 12.7, 32000 x 2048 23.6 / 21.4, x 4096 43.9 / 40.6, 128256 x 4096 164 / 150 (four rows a wave: 14.6, 24.2, 41.8, 156).
// gate | up: eight waves with a pair each, but four up to 2048 rows of more than 1024 columns, a workgroup of four waves a CU (four / eight: 2048 x 1024 3.6 / 3.5, x 2048
// 4.5 / 4.7, x 3072 5.6 / 6.1; 2560 x 2048 5.2 / 4.9, 16384 x 2048 13.3 / 12.8).
template <int IN, int OUT>
inline void launch_gemv1_bf16(hipStream_t st, crabml_hip_device::ProfRec* rec, const GemvBf16& a) {
  constexpr bool NARROW = OUT == GEMV_OUT_RESIDUAL || OUT == GEMV_OUT_STREAMS;  // (as many rows as the model is wide)
  if constexpr (OUT == GEMV_OUT_GLU) {
    if (a.K <= 512)
      launch_gemv_bf16_t<8, 1, 2, 1, IN, OUT>(st, rec, a);
    else if (a.K <= 1024)
      launch_gemv_bf16_t<8, 1, 2, 2, IN, OUT>(st, rec, a);
    else if (a.N > 2048)
      launch_gemv_bf16_t<8, 1, 2, 4, IN, OUT>(st, rec, a);
    else
      launch_gemv_bf16_t<4, 1, 2, 4, IN, OUT>(st, rec, a);
    return;
  } else {
    if constexpr (!NARROW) {
      if (a.K <= 512 && a.N >= 16384) return launch_gemv_bf16_t<8, 1, 4, 1, IN, OUT>(st, rec, a);
      if (a.K <= 512 && a.N > 8192) return launch_gemv_bf16_t<8, 1, 2, 1, IN, OUT>(st, rec, a);
      if (a.K < 2048 && a.N > 8192)
        return a.K <= 1024 ? launch_gemv_bf16_t<8, 1, 2, 2, IN, OUT>(st, rec, a) : launch_gemv_bf16_t<8, 1, 2, 4, IN, OUT>(st, rec, a);
    }
    if (a.K <= 512)
      launch_gemv_bf16_t<8, 1, 1, 1, IN, OUT>(st, rec, a);
    else if (a.K <= 1024)
      launch_gemv_bf16_t<8, 1, 1, 2, IN, OUT>(st, rec, a);
    else if (a.N <= 1024 && a.K >= 4096)
      launch_gemv_bf16_t<4, 1, 1, 8, IN, OUT>(st, rec, a);
    else if (a.K > 4096 && (a.N <= 2048 || a.K >= 8192))
      launch_gemv_bf16_t<8, 1, 1, 8, IN, OUT>(st, rec, a);
    else if (a.N <= 1024 || (a.N >= 16384 && a.K <= 4096 && IN != GEMV_IN_RMSV))
      launch_gemv_bf16_t<4, 1, 1, 4, IN, OUT>(st, rec, a);
    else
      launch_gemv_bf16_t<8, 1, 1, 4, IN, OUT>(st, rec, a);
  }
}
// Two rows: the same (2048 x 512 3.95 / 3.6, 1280 x 4096 5.5 / 4.8, 2048 x 8192 9.5 / 8.4, 8192 x 4096 14.3 / 13.25), but two rows of weights a wave where there are more than
// 4096 of up to 1024 columns or more than 2048 of up to 2048 (a row each / two, four waves: 4096 x 1024 4.97 / 5.08, 8192 x 1024 6.9 / 6.7, 32000 x 1024 17.9 / 14.8; 2048 x 2048
// 4.9 / 5.15, 3648 x 2048 6.36 / 6.35, 32000 x 2048 24.3 / 23.0); where they are more and longer and the rhs is staged with a gain per element, two each in eight waves (3136 x
// 2560 7.6 / 6.9, 3136 x 4096 9.1 / 8.6, 32000 x 4096 46.7 / 41.8; 2048 x 4096 6.6 / 7.85).  gate | up: four waves up to 2048 rows, else eight (2048 x 2048 5.1 / 5.6,
// 2048 x 1024 4.25 / 4.4, 2560 x 2048 6.05 / 5.8, 16384 x 1024 9.9 / 9.4, x 2048 15.5 / 14.5).
template <int IN, int OUT>
inline void launch_gemv2_bf16(hipStream_t st, crabml_hip_device::ProfRec* rec, const GemvBf16& a) {
  if constexpr (OUT == GEMV_OUT_GLU) {
    if (a.N > 2048)
      a.K <= 1024 ? launch_gemv_bf16_t<8, 2, 2, 2, IN, OUT>(st, rec, a) : launch_gemv_bf16_t<8, 2, 2, 4, IN, OUT>(st, rec, a);
    else
      a.K <= 1024 ? launch_gemv_bf16_t<4, 2, 2, 2, IN, OUT>(st, rec, a) : launch_gemv_bf16_t<4, 2, 2, 4, IN, OUT>(st, rec, a);
  } else {
    if constexpr (IN == GEMV_IN_RMSV) {
      if (a.K > 2048 && a.N > 2048) return launch_gemv_bf16_t<8, 2, 2, 4, IN, OUT>(st, rec, a);
    }
    if (a.K <= 1024 && a.N > 4096)
      launch_gemv_bf16_t<4, 2, 2, 2, IN, OUT>(st, rec, a);
    else if (a.K <= 1024)
      launch_gemv_bf16_t<8, 2, 1, 2, IN, OUT>(st, rec, a);
    else if (a.K <= 2048 && a.N > 2048)
      launch_gemv_bf16_t<4, 2, 2, 4, IN, OUT>(st, rec, a);
    else
      launch_gemv_bf16_t<8, 2, 1, 4, IN, OUT>(st, rec, a);
  }
}
// Eight rows (matmul_vec): the next steps' requests together, behind the products; step by step 8192 x 2048 15.1 us against 9.9, 8192 x 8192 49.1 / 32.0, 32000 x 2048
// 49.4 / 39.4.  Four rows: step by step 8.0 -> 7.4, 26.3 -> 23.6, 26.6 -> 23.7.
// rows of the rhs that share one pass over the weights: as many as there are, up to 8; in front of and behind anything else two (a step's linears have no more here)
template <int IN, int OUT>
inline void launch_gemv_bf16(hipStream_t st, crabml_hip_device::ProfRec* rec, const GemvBf16& a) {
  if (a.nb <= 1) return launch_gemv1_bf16<IN, OUT>(st, rec, a);
  if constexpr (IN == GEMV_IN_PLAIN && OUT == GEMV_OUT_STORE) {
    if (a.nb > 4) return launch_gemv_bf16_t<4, 8, 2, 2, IN, OUT, false>(st, rec, a);
    if (a.nb > 2) return launch_gemv_bf16_t<4, 4, 2, 4, IN, OUT>(st, rec, a);
  }
  launch_gemv2_bf16<IN, OUT>(st, rec, a);
}

}  // namespace crabml_hip
