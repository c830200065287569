// prefill_rows.hpp -- row kernels of the FAST prompt pass that also leave the row's pre-scaled f16 plane B' for the weight GEMM that
// reads it next (gemm_f16w.hip; slot orders: f16w_rows.hpp): the same arithmetic as the kernels they wrap, one k_rows_to_f16 launch
// fewer per GEMM.  B' is bit for bit what k_rows_to_f16 makes from the finished planes.
#pragma once
#include "f16w_rows.hpp"
#include "fused_common.hpp"
#include "fused_ffn.hpp"

namespace crabml_hip {

// Residual add (+ the k pieces of the GEMM that made the addend: piece 0 in addv, the others added to it first, in piece order -- k_addn_f32's arithmetic) +
// RMSNorm + quantize + the row's B' (xh, nullable), a workgroup of 256 threads per row.  A thread has NJ groups of four consecutive elements, 1024 apart, so
// that a wave's requests and stores are whole lines, a 32-element chunk is 8 lanes and a super-block of 256 a wave; everything that the row needs is asked
// for at once, the pieces of all groups together.  Arithmetic = norm_quant_block's and the quantizers', bit for bit: a chunk's squares from -0.0 in
// element order, handed from lane to lane (half: rows 0..15 and 16..31 separately, then added -- the fast step's order; else one 32-element scan,
// rms_norm.rs:35-38); the chunk sums as there (half: 64 per round through wave_sum_f32, rounds in order; else strictly in chunk order), by every wave for
// itself; (x / rms) * w.  What bounds it: the row's traffic through memory behind one chain of two round trips, and its divisions.  Us a launch, a thread on
// sixteen consecutive elements or 1024 threads with the row in LDS / so: 512 rows of 4096 to Q8_0 12.4 / 11.1, 1024 to Q8_K 22.5 / 14.5, one to Q8_K 6.0 / 5.7;
// a Q4_K prompt of four layers of width 2048, the launches one by one / so: 4 rows 426 / 380, 33 rows 475 / 420, 190 rows 520 / 458.
template <int NJ, int QT>
__global__ __launch_bounds__(256) void k_norm_quant_rows(float* __restrict__ x, const float* __restrict__ addv, const float* __restrict__ w, int cols, float eps,
                                                        char* __restrict__ planes, size_t row_stride, size_t off_d, size_t off_aux, size_t off_p, int half,
                                                        unsigned short* __restrict__ xh, int xh_order, const float* __restrict__ parts, size_t pstride, int nparts) {
  __shared__ float cs_lds[NJ * 32];
  const int tid = threadIdx.x, lane = tid & 63, n4 = cols / 4;
  const size_t r = blockIdx.x;
  f32x4* xr = (f32x4*)(x + r * cols);
  const f32x4* ar = (const f32x4*)(addv ? addv + r * cols : x + r * cols);
  f32x4 xv[NJ], av[NJ], wv[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int i = j * 256 + tid < n4 ? j * 256 + tid : n4 - 1;
    av[j] = ar[i];
    xv[j] = xr[i];
    wv[j] = ((const f32x4*)w)[i];
  }
  for (int s = 0; s < nparts; s++) {
    const f32x4* pr = (const f32x4*)(parts + (size_t)s * pstride + r * cols);
    f32x4 pv[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) pv[j] = pr[j * 256 + tid < n4 ? j * 256 + tid : n4 - 1];
#pragma unroll
    for (int j = 0; j < NJ; j++) av[j] = av[j] + pv[j];
  }
  const int last = half ? 3 : 7;  // lanes that a scan goes through, less one
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int i = j * 256 + tid;
    if (addv) {
      xv[j] = av[j] + xv[j];  // x = matmul_out + x (llama2.rs:266 / :636)
      if (i < n4) xr[i] = xv[j];
    }
    const float t = quad_square_scan(xv[j], lane, last);
    const float low = dpp_f<0x114>(t);  // (row_shr:4: rows 0..15's)
    if ((lane & 7) == 7 && i < n4) cs_lds[i >> 3] = half ? low + t : t;
  }
  __syncthreads();
  const float rms = sqrtf(chunk_sums(cs_lds, cols / 32, lane, half) / (float)cols + eps);
  char* p = planes + r * row_stride;
  unsigned short* xo = xh + r * (size_t)cols;
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int i = j * 256 + tid;
    if (j * 256 + (tid & ~63) >= n4) break;  // (wave-uniform)
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = (xv[j][e] / rms) * wv[j][e];
    if constexpr (QT == CRABML_HIP_Q8_K) {  // (whole waves: cols is a multiple of 256)
      const int sb = i >> 6;
      const Q8KLane o = q8k_wave_quant(v, lane);
      ((unsigned*)p)[i] = o.packed;
      q8k_store_class_major((signed char*)(p + off_p) + sb * 256, lane, o.packed);
      if ((lane & 3) == 0) ((short*)(p + off_aux))[i >> 2] = (short)o.quad_sum;
      if (lane == 0) ((float*)(p + off_d))[sb] = o.d;
      if (xh) f16w_store_q8k(xo, xh_order, sb, lane, o.packed, o.d);
    } else {
      constexpr bool Q81 = QT == CRABML_HIP_Q8_1;
      const QLane4 o = quant_quad8<Q81>(v);
      if (i >= n4) continue;  // (whole chunks)
      ((unsigned*)p)[i] = o.packed;
      if ((lane & 7) == 0) {
        ((unsigned short*)(p + off_d))[i >> 3] = o.d;
        store_qaux<Q81>((void*)(p + off_aux), i >> 3, o.aux);
      }
      if (xh) f16w_store4(xo + (i >> 3) * 32 + 8 * (i & 3) + 4 * (i >> 2 & 1), o.packed, h2f(o.d));
    }
  }
}
template <int QT, typename... A>
inline void launch_norm_quant_rows(hipStream_t st, size_t rows, int cols, A... a) {
  if (cols <= 1024)
    k_norm_quant_rows<1, QT><<<(unsigned)rows, 256, 0, st>>>(a...);
  else if (cols <= 2048)
    k_norm_quant_rows<2, QT><<<(unsigned)rows, 256, 0, st>>>(a...);
  else if (cols <= 4096)
    k_norm_quant_rows<4, QT><<<(unsigned)rows, 256, 0, st>>>(a...);
  else if (cols <= 8192)
    k_norm_quant_rows<8, QT><<<(unsigned)rows, 256, 0, st>>>(a...);
  else
    k_norm_quant_rows<12, QT><<<(unsigned)rows, 256, 0, st>>>(a...);
}

// k_gateup_epi_quant (h = silu(g) * u quantized straight into the rows' Q8_0 / Q8_1 planes) + the rows' B' (order 0)
template <bool Q81>
__global__ __launch_bounds__(256) void k_gateup_epi_quant_h(const float* __restrict__ g, const float* __restrict__ u,
                                                            const unsigned short* __restrict__ exp_tab, int hidden, char* __restrict__ planes,
                                                            size_t row_stride, size_t off_d, size_t off_aux, unsigned short* __restrict__ xh) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;  // hidden % 32 == 0: half-waves are all-live or all-dead
  const size_t r = blockIdx.y;
  const bool live = i < hidden;
  const float h = live ? silu_mul(g[r * hidden + i], u[r * hidden + i], exp_tab) : 0.0f;
  const QLane o = quant_lane32<Q81>(h, live);
  if (!live) return;
  char* p = planes + r * row_stride;
  ((signed char*)p)[i] = o.q;
  if ((threadIdx.x & 31) == 0) {
    ((unsigned short*)(p + off_d))[i >> 5] = o.d;
    store_qaux<Q81>((void*)(p + off_aux), i >> 5, o.aux);
  }
  xh[r * (size_t)hidden + (i & ~31) + f16w_slot_of_elem(i & 31)] = f16w_value((int)o.q, h2f(o.d));
}

}  // namespace crabml_hip
