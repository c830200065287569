// quantize.hip -- on-the-fly activation quantization for matmul_vec's rhs.
//
// Replaces CpuTensorBuf::quantize (crabml-core/src/cpu/buf/api.rs:195-228) as called from
// gemv_dense_2d_2d (crabml-core/src/cpu/primitives/matmul_vec.rs:37-40).  The arithmetic follows the
// reference, NOT ggml:
//   Q8_0  d = max|x| / 127 ; q = trunc(x / d)  (true division; simd cast: NaN -> 0)   buf_q8_0.rs:87-134
//   Q8_1  d = max|x| / 127 ; q = trunc(clamp(x / d, -128, 127)) (NaN -> -128) ; s = f16(d * sum q)
//                                                                                    buf_q8_1.rs:90-129
//   Q8_K  mx = first element of max |x| ; scale = -128 / mx ; q = min(round_half_away(scale * x), 127) ;
//         d = 1 / scale ; bsums over 16                                              buf_q8_k.rs:84-131
// Output goes to "planes" (see common.hpp).  All outputs are bit-identical to the reference's blocks
// (tests/test_hip_quantize.py compares the bytes).
#include "devutil.hpp"
#include "f16w_rows.hpp"
#include "kernels.hpp"

namespace crabml_hip {

// eight lanes per block, four consecutive elements each: a wave's request and its stores are whole lines (a lane per element: 512 rows of 4096 with B'
// 8.6 us)
template <bool Q81>
__global__ __launch_bounds__(256) void k_quantize_q8(const float* __restrict__ x, char* __restrict__ planes, size_t off_d, size_t off_aux, size_t nblocks,
                                                     size_t row_elems, size_t row_bytes, unsigned short* __restrict__ xh) {
  // blockIdx.y: row of a batch (x rows of row_elems floats; one set of planes every row_bytes bytes)
  // xh (nullable): the row's pre-scaled f16 plane for the fast prompt pass's GEMM (f16w_rows.hpp), written next to the planes
  char* p = planes + blockIdx.y * row_bytes;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, blk = i >> 3;
  const bool live = blk < nblocks;
  const QLane4 o = quant_quad8<Q81>(((const f32x4*)(x + blockIdx.y * row_elems))[live ? i : 0]);
  if (!live) return;  // (whole blocks)
  ((unsigned*)p)[i] = o.packed;
  if ((i & 7) == 0) {
    ((unsigned short*)(p + off_d))[blk] = o.d;
    if constexpr (Q81)
      ((unsigned short*)(p + off_aux))[blk] = (unsigned short)o.aux;
    else
      ((int*)(p + off_aux))[blk] = o.aux;
  }
  if (xh) f16w_store4(xh + blockIdx.y * row_elems + blk * 32 + 8 * (i & 3) + 4 * (i >> 2 & 1), o.packed, h2f(o.d));
}

// one wave per 256-element super-block, 4 consecutive elements per lane
__global__ __launch_bounds__(256) void k_quantize_q8_k(const float* __restrict__ x, signed char* __restrict__ q,
                                                       float* __restrict__ d, short* __restrict__ bsums, signed char* __restrict__ qp,
                                                       size_t nblocks, size_t row_elems, size_t row_bytes, unsigned short* __restrict__ xh, int xh_order) {
  x += blockIdx.y * row_elems;
  q += blockIdx.y * row_bytes;
  qp += blockIdx.y * row_bytes;
  d = (float*)((char*)d + blockIdx.y * row_bytes);
  bsums = (short*)((char*)bsums + blockIdx.y * row_bytes);
  const int lane = threadIdx.x & 63;
  size_t blk = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (blk >= nblocks) return;  // whole wave exits together
  const f32x4 v = *(const f32x4*)(x + blk * 256 + lane * 4);
  const Q8KLane o = q8k_wave_quant(v, lane);  // devutil.hpp
  *(unsigned*)(q + blk * 256 + lane * 4) = o.packed;
  q8k_store_class_major(qp + blk * 256, lane, o.packed);  // the plane the Q4_K kernels read
  if ((lane & 3) == 0) bsums[blk * 16 + (lane >> 2)] = (short)o.quad_sum;
  if (lane == 0) d[blk] = o.d;
  if (xh) f16w_store_q8k(xh + blockIdx.y * row_elems, xh_order, (int)blk, lane, o.packed, o.d);  // (xh_order 1 / 2: the k-slot order of Q4_K / Q6_K weights)
}

__global__ __launch_bounds__(256) void k_quantize_f16(const float* __restrict__ x, unsigned short* __restrict__ h,
                                                      size_t n, size_t row_bytes) {
  x += blockIdx.y * n;
  h = (unsigned short*)((char*)h + blockIdx.y * row_bytes);
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) h[i] = f2h(x[i]);
}

void launch_quantize_act(hipStream_t st, uint32_t qtype, const float* x, size_t n, void* planes) {
  launch_quantize_act_rows(st, qtype, x, 1, n, planes);
}
// xh (nullable; Q8_0 / Q8_1 / Q8_K): (rows, n) halfs -- the rows' pre-scaled f16 planes in k-slot order `xh_order` (gemm_f16w_order of the
// weight format that will read them), bit for bit what launch_rows_to_f16 makes from the finished planes
// rows vectors of n elements each -> rows sets of planes, act_layout(qtype, n).total bytes apart (the batched rhs of
// launch_gemv)
void launch_quantize_act_rows(hipStream_t st, uint32_t qtype, const float* x, size_t rows, size_t n, void* planes, void* xh, int xh_order) {
  if (n == 0 || rows == 0) return;
  ActLayout al = act_layout(qtype, n);
  const unsigned ry = (unsigned)rows;
  char* p = (char*)planes;
  switch (qtype) {
    case CRABML_HIP_Q8_0:
    case CRABML_HIP_Q8_1: {
      const size_t nb = n / 32;
      const dim3 grid((unsigned)((nb * 8 + 255) / 256), ry);
      if (qtype == CRABML_HIP_Q8_0)
        k_quantize_q8<false><<<grid, 256, 0, st>>>(x, p, al.off_d, al.off_aux, nb, n, al.total, (unsigned short*)xh);
      else
        k_quantize_q8<true><<<grid, 256, 0, st>>>(x, p, al.off_d, al.off_aux, nb, n, al.total, (unsigned short*)xh);
      break;
    }
    case CRABML_HIP_Q8_K: {
      size_t nb = n / 256;
      unsigned grid = (unsigned)((nb + 3) / 4);
      k_quantize_q8_k<<<dim3(grid, ry), 256, 0, st>>>(x, (signed char*)p, (float*)(p + al.off_d), (short*)(p + al.off_aux),
                                                      (signed char*)(p + al.off_p), nb, n, al.total, (unsigned short*)xh, xh_order);
      break;
    }
    case CRABML_HIP_F16: {
      unsigned grid = (unsigned)((n + 255) / 256);
      k_quantize_f16<<<dim3(grid, ry), 256, 0, st>>>(x, (unsigned short*)p, n, al.total);
      break;
    }
    default: break;
  }
}

}  // namespace crabml_hip
