// fused_f16.hpp -- the fast decode step's linears over F16 weights, with the row operations around them folded into their two ends.
//
// Per layer: [norm + q | k | v + rope + append], attention, [wo + residual], [norm + gate | up + SiLU * mul], [ffn_down + residual] -- four
// launches of this kernel and the attention's, where the per-op segments take eighteen, most of them 2-5 us of nothing but launch.
//
// Mapping: a wave owns R weight rows and strides k 512 elements at a time (8 per lane: one aligned 16-byte request per row), UN steps in
// flight; the first requests go out before the rhs is looked at.  The rhs is what the reference multiplies by (buf/api.rs:142-159: the row
// rounded to f16): a workgroup of eight waves (four: launch_step_f16) normalizes (x / rms) * w, or rounds, the whole row into LDS itself -- 2 bytes per element, read
// back as contiguous 16-byte pieces -- which is 8-16 KB from L2 per workgroup beside its 16-64 KB of weights and hides behind them.
// ffn_down's rhs leaves the gate | up launch as f16 already and is read from L2 in place.  Products are exact in f32 (v_fma_mix_f32), sums
// f32.  Bound: the weights' bytes, plus a launch's ramp.
#pragma once
#include "fused_common.hpp"

namespace crabml_hip {

enum { F16_IN_NORM = 0, F16_IN_ROUND = 1, F16_IN_HALF = 2 };
enum { F16_OUT_QKV = 0, F16_OUT_RES = 1, F16_OUT_GU = 2, F16_OUT_STORE = 3 };

struct StepF16 {
  const unsigned short* w[3] = {nullptr, nullptr, nullptr};  // q, k, v / gate, up / the matrix
  int m = 0;                    // rows: of all three (QKV), of one of the two (GU), of the matrix
  int k = 0;                    // a multiple of 8
  const float* x = nullptr;     // NORM, ROUND: the f32 row
  const float* gain = nullptr;  // NORM
  float eps = 0.f;
  const unsigned short* x16 = nullptr;  // HALF
  float* out = nullptr;                 // RES (+=), STORE
  unsigned short* h16 = nullptr;        // GU
  const unsigned short* exp_tab = nullptr;
};

// WV: waves of a workgroup; NIT: rhs pieces of 8 elements a thread holds while the norm is taken (k <= NIT * WV * 512)
template <int WV, int R, int UN, int NIT, int IN, int OUT>
__global__ __launch_bounds__(64 * WV) void k_step_f16(const StepF16 a, const QkvEpi e) {
  extern __shared__ __attribute__((aligned(16))) unsigned short rhs[];  // [k], NORM and ROUND
  __shared__ float red[WV];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg();
  const int unit = blockIdx.x * WV + wave;  // this wave's rows: R unit .. (GU: R / 2 of either matrix)
  const unsigned short* wr[R];
  bool live[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    if constexpr (OUT == F16_OUT_GU) {
      const int row = unit * (R / 2) + r % (R / 2);
      live[r] = row < a.m;
      wr[r] = a.w[r / (R / 2)] + (size_t)(live[r] ? row : a.m - 1) * a.k;
    } else {
      int row = unit * R + r;
      live[r] = row < a.m;
      row = live[r] ? row : a.m - 1;
      const unsigned short* base = a.w[0];
      if constexpr (OUT == F16_OUT_QKV) {
        base = row < e.dim ? a.w[0] : row < e.dim + e.kv_dim ? a.w[1] : a.w[2];
        row -= row < e.dim ? 0 : row < e.dim + e.kv_dim ? e.dim : e.dim + e.kv_dim;
      }
      wr[r] = base + (size_t)row * a.k;
    }
  }
  i32x4 wv[UN][R], xv[UN];
  auto request = [&](int k0) {
#pragma unroll
    for (int u = 0; u < UN; u++) {
      int i = k0 + u * 512 + lane * 8;
      i = i < a.k ? i : 0;  // (a lane past the end requests the row's start and never uses it)
#pragma unroll
      for (int r = 0; r < R; r++) wv[u][r] = __builtin_nontemporal_load((const i32x4*)(wr[r] + i));
      if constexpr (IN == F16_IN_HALF) xv[u] = *(const i32x4*)(a.x16 + i);
    }
  };
  request(0);
  QkvPre pre{};
  if constexpr (OUT == F16_OUT_QKV) pre = qkv_preload_nb(e, live[0] ? unit * R : 0);
  float old[R];
  if constexpr (OUT == F16_OUT_RES) {
#pragma unroll
    for (int r = 0; r < R; r++) old[r] = a.out[live[r] ? unit * R + r : 0];
  }
  if constexpr (IN != F16_IN_HALF) {
    f32x4 v[NIT][2], gn[NIT][2];
#pragma unroll
    for (int it = 0; it < NIT; it++) {
      const int i = (it * (64 * WV) + tid) * 8, at = i < a.k ? i : 0;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        v[it][h] = *(const f32x4*)(a.x + at + 4 * h);
        if constexpr (IN == F16_IN_NORM) gn[it][h] = *(const f32x4*)(a.gain + at + 4 * h);
      }
    }
    float rms = 1.f;
    if constexpr (IN == F16_IN_NORM) {
      float sq = 0.f;
#pragma unroll
      for (int it = 0; it < NIT; it++)
        if ((it * (64 * WV) + tid) * 8 < a.k) {
#pragma unroll
          for (int h = 0; h < 2; h++)
#pragma unroll
            for (int c = 0; c < 4; c++) sq = __builtin_fmaf(v[it][h][c], v[it][h][c], sq);
        }
      sq = wave_sum_f32(sq);
      if (lane == 0) red[wave] = sq;
      __syncthreads();
      sq = 0.f;
#pragma unroll
      for (int w = 0; w < WV; w += 4) sq += (red[w] + red[w + 1]) + (red[w + 2] + red[w + 3]);
      rms = sqrtf(sq / (float)a.k + a.eps);
    }
#pragma unroll
    for (int it = 0; it < NIT; it++) {
      const int i = (it * (64 * WV) + tid) * 8;
      if (i < a.k) {
        unsigned short t[8];
#pragma unroll
        for (int c = 0; c < 8; c++) t[c] = f2h(IN == F16_IN_NORM ? (v[it][c / 4][c % 4] / rms) * gn[it][c / 4][c % 4] : v[it][c / 4][c % 4]);
        i32x4 p;
        __builtin_memcpy(&p, t, 16);
        *(i32x4*)(rhs + i) = p;
      }
    }
    __syncthreads();
  }
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; r++) acc[r] = 0.f;
  for (int k0 = 0; k0 < a.k; k0 += UN * 512) {
    i32x4 wc[UN][R], xc[UN];
#pragma unroll
    for (int u = 0; u < UN; u++) {
#pragma unroll
      for (int r = 0; r < R; r++) wc[u][r] = wv[u][r];
      if constexpr (IN == F16_IN_HALF) xc[u] = xv[u];
    }
    if (k0 + UN * 512 < a.k) request(k0 + UN * 512);
#pragma unroll
    for (int u = 0; u < UN; u++) {
      const int i = k0 + u * 512 + lane * 8;
      if (i < a.k) {
        if constexpr (IN != F16_IN_HALF) xc[u] = *(const i32x4*)(rhs + i);
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] = dot_f16x8(wc[u][r], xc[u], acc[r]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++) acc[r] = wave_sum_f32(acc[r]);
  if (lane != 0) return;
  if constexpr (OUT == F16_OUT_QKV) {
    static_assert(OUT != F16_OUT_QKV || R == 2, "a wave holds the pair that is rotated");
    if (live[0]) qkv_epilogue(e, pre, unit * R, acc[0], acc[1]);
  } else if constexpr (OUT == F16_OUT_GU) {
#pragma unroll
    for (int r = 0; r < R / 2; r++)
      if (live[r]) a.h16[unit * (R / 2) + r] = f2h(silu_mul(acc[r], acc[r + R / 2], a.exp_tab));
  } else {
#pragma unroll
    for (int r = 0; r < R; r++)
      if (live[r]) a.out[unit * R + r] = OUT == F16_OUT_RES ? acc[r] + old[r] : acc[r];
  }
}

}  // namespace crabml_hip
