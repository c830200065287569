// f16w_rows.hpp -- where an activation element sits in the pre-scaled f16 planes B' that the fast prompt pass's weight GEMM reads
// (gemm_f16w.hip: xh[row][k] halfs in the GEMM's k-slot order).  k_rows_to_f16 makes B' from finished planes; the row kernels of the
// pass that quantize a row (quantize.hip, prefill_rows.hpp) write it themselves with these, one launch fewer per GEMM.
#pragma once
#include "devutil.hpp"

namespace crabml_hip {

// order 0 (Q8_0 / Q8_1 rows; Q4_0, Q8_0, Q4_1 weights): slot of element j of a 32-element block -- the inverse of f16w_slot_elem
__device__ __forceinline__ int f16w_slot_of_elem(int j) {
  const int hi = j >> 4, s = (j >> 2) & 3, r = j & 3;
  return 8 * s + 4 * hi + ((r >> 1) | ((r & 1) << 1));
}
// orders 1 (Q4_K weights) / 2 (Q6_K weights), Q8_K rows: element E of super-block sb sits at half (4 cc + g) * 32 + 8 s + 4 hi + {0, 2, 1, 3}[k] of the row, with
//   order 1: l = E % 8, k = E / 8 % 4, hi = E / 32 % 2, g = E / 64, s = l % 4, cc = 2 sb + l / 4
//   order 2: k = E % 4, s = E / 4 % 4, g = E / 16 % 4, hi = E / 64 % 2, cc = 2 sb + E / 128
// order 0: inside a block, slot 8 s + e (s = 0..3 = the dword of the weight block the slot pairs with) holds element
//   e = 0, 1: 4 s, 4 s + 2     e = 2, 3: 4 s + 1, 4 s + 3     e = 4, 5: 16 + 4 s, 16 + 4 s + 2     e = 6, 7: 16 + 4 s + 1, 16 + 4 s + 3
// -- the order in which unpack_q4_0_f16 takes the nibbles out of a dword (two masks per packed pair, no byte permute)
__device__ __forceinline__ int f16w_slot_elem(int slot) {
  const int s = slot >> 3, e = slot & 7;
  return (e >= 4 ? 16 : 0) + 4 * s + ((e >> 1) & 1) + 2 * (e & 1);
}
// one 8-slot group t = 4 kb + s of a row's B' from its FINISHED planes p (q | d at off_d): xrow[kb * 32 + 8 s ..]
template <int ORDER>
__device__ __forceinline__ void rows_to_f16_piece(const char* __restrict__ p, size_t off_d, int t, unsigned short* __restrict__ xrow) {
  const int kb = t >> 2, s = t & 3;
  float d;
  const signed char* q;
  int at[8];
  if constexpr (ORDER == 2) {
    const int cc = kb >> 2, g = kb & 3, sb = cc >> 1;
    d = ((const float*)(p + off_d))[sb];
    q = (const signed char*)p + sb * 256 + 128 * (cc & 1) + 32 * (g >> 1) + 16 * (g & 1) + 4 * s;
#pragma unroll
    for (int e = 0; e < 8; e++) at[e] = (e >= 4 ? 64 : 0) + ((e >> 1) & 1) + 2 * (e & 1);
  } else if constexpr (ORDER == 1) {
    const int cc = kb >> 2, g = kb & 3, sb = cc >> 1, l = 4 * (cc & 1) + s;
    d = ((const float*)(p + off_d))[sb];
    q = (const signed char*)p + sb * 256 + 64 * g;
#pragma unroll
    for (int e = 0; e < 8; e++) at[e] = (e >= 4 ? 32 : 0) + 8 * (((e >> 1) & 1) + 2 * (e & 1)) + l;
  } else {
    d = h2f(((const unsigned short*)(p + off_d))[kb]);
    q = (const signed char*)p + kb * 32;
#pragma unroll
    for (int e = 0; e < 8; e++) at[e] = f16w_slot_elem(8 * s + e);
  }
  unsigned short o[8];
#pragma unroll
  for (int e = 0; e < 8; e++) o[e] = f2h((float)q[at[e]] * d);  // (Q8_0: 7-bit x 11-bit, exact in f32, one rounding; Q8_K: f32 d, two)
  *(i32x4*)(xrow + kb * 32 + 8 * s) = i32x4{(int)(o[0] | ((unsigned)o[1] << 16)), (int)(o[2] | ((unsigned)o[3] << 16)),
                                            (int)(o[4] | ((unsigned)o[5] << 16)), (int)(o[6] | ((unsigned)o[7] << 16))};
}
// the f16 value of a quant: q * d in f32 (Q8_0 / Q8_1: d is the STORED f16 scale -- exact product, one rounding), rounded once
__device__ __forceinline__ unsigned short f16w_value(int q, float d) { return f2h((float)q * d); }

// four of a row's B' values from the quants 0 .. 3 of a dword that stand 0, 2, 1, 3 there
__device__ __forceinline__ void f16w_store4(unsigned short* at, unsigned quants, float d) {
  const unsigned short v0 = f16w_value((int)(signed char)(quants & 0xffu), d), v1 = f16w_value((int)(signed char)((quants >> 8) & 0xffu), d);
  const unsigned short v2 = f16w_value((int)(signed char)((quants >> 16) & 0xffu), d), v3 = f16w_value((int)(signed char)(quants >> 24), d);
  *(unsigned long long*)at = (unsigned long long)(v0 | ((unsigned)v2 << 16)) | ((unsigned long long)(v1 | ((unsigned)v3 << 16)) << 32);
}
// B' of super-block sb from a wave's quantizer (q8k_wave_quant: lane has the quants of elements 4 lane .. 4 lane + 3): their places above, eight bytes a
// lane -- order 2 keeps four consecutive elements together, order 1 the four of a class, which is what the class-major dword holds
__device__ __forceinline__ void f16w_store_q8k(unsigned short* __restrict__ xrow, int order, int sb, int lane, unsigned packed, float d) {
  if (order == 1) {
    const int l = (lane & 1) * 4 + ((lane >> 1) & 3);  // (the dword's class: q8k_class_major_at)
    f16w_store4(xrow + (4 * (2 * sb + (l >> 2)) + (lane >> 4)) * 32 + 8 * (l & 3) + 4 * (lane >> 3 & 1), q8k_class_major(lane, packed), d);
  } else {
    f16w_store4(xrow + (4 * (2 * sb + (lane >> 5)) + 2 * (lane >> 3 & 1) + (lane >> 2 & 1)) * 32 + 8 * (lane & 3) + 4 * (lane >> 4 & 1), packed, d);
  }
}

}  // namespace crabml_hip
