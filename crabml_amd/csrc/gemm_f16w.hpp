// gemm_f16w.hpp -- what the kernels of the fast prompt pass's weight GEMM share (gemm_f16w.hip, gemm_f16w_wide.hip): the operands'
// conversion to f16 fragments, the matrices of a launch, and h = silu(g) * u quantized where it was computed.
#pragma once
#include "devutil.hpp"
#include "f16w_rows.hpp"
#include "kernels.hpp"

namespace crabml_hip {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// one dword of a Q4_0 block (quant bytes 4 s .. 4 s + 3: low nibbles = elements 4 s .., high nibbles = 16 + 4 s ..; buf_q4_0.rs:24-33)
// -> the lane's eight f16 k-slots (q - 8) * d.  0x6400 | n is the f16 number 1024 + n; -1032 makes it n - 8 exactly.
// (x & 0x000F000F) | 0x64006400 as ONE v_and_or_b32: a VOP3 instruction takes a single scalar / literal operand, so the compiler
// splits it unless one constant sits in a VGPR -- `magic` (loop-invariant, one register)
__device__ __forceinline__ unsigned and_or_magic(unsigned x, unsigned magic) {
  unsigned r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(0x000F000Fu), "v"(magic));
  return r;
}
__device__ __forceinline__ f16x8 unpack_q4_0_f16(unsigned w, f16x2 d2, unsigned magic) {
  const f16x2 bias = {(_Float16)-1032.0f, (_Float16)-1032.0f};
  const unsigned u0 = and_or_magic(w, magic), u1 = and_or_magic(w >> 8, magic);
  const unsigned u2 = and_or_magic(w >> 4, magic), u3 = and_or_magic(w >> 12, magic);
  const f16x2 p0 = (__builtin_bit_cast(f16x2, u0) + bias) * d2, p1 = (__builtin_bit_cast(f16x2, u1) + bias) * d2;
  const f16x2 p2 = (__builtin_bit_cast(f16x2, u2) + bias) * d2, p3 = (__builtin_bit_cast(f16x2, u3) + bias) * d2;
  return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// Q8_0: the bytes of a dword as f16 (b ^ 0x80 = b + 128 unsigned; 0x6400 | u = 1024 + u; -1152 makes it b exactly), pairs (b0, b2), (b1, b3)
__device__ __forceinline__ unsigned and_or_magic8(unsigned x, unsigned magic) {
  unsigned r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(0x00FF00FFu), "v"(magic));
  return r;
}
__device__ __forceinline__ f16x8 unpack_q8_0_f16(unsigned w0, unsigned w1, f16x2 d2, unsigned magic) {
  const f16x2 bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
  const unsigned x0 = w0 ^ 0x80808080u, x1 = w1 ^ 0x80808080u;
  const unsigned u0 = and_or_magic8(x0, magic), u1 = and_or_magic8(x0 >> 8, magic);
  const unsigned u2 = and_or_magic8(x1, magic), u3 = and_or_magic8(x1 >> 8, magic);
  const f16x2 p0 = (__builtin_bit_cast(f16x2, u0) + bias) * d2, p1 = (__builtin_bit_cast(f16x2, u1) + bias) * d2;
  const f16x2 p2 = (__builtin_bit_cast(f16x2, u2) + bias) * d2, p3 = (__builtin_bit_cast(f16x2, u3) + bias) * d2;
  return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}
// Q4_K: one class dword of the lane's pair; cs = {d sc_lo, -dmin m_lo, d sc_hi, -dmin m_hi}, each in both halves
struct Q4KF16Consts {
  f16x2 c_lo, o_lo, c_hi, o_hi;
};
__device__ __forceinline__ f16x8 unpack_q4_k_f16(unsigned w, const Q4KF16Consts& cs, unsigned magic) {
  const f16x2 bias = {(_Float16)-1024.0f, (_Float16)-1024.0f};
  const unsigned u0 = and_or_magic(w, magic), u1 = and_or_magic(w >> 8, magic);
  const unsigned u2 = and_or_magic(w >> 4, magic), u3 = and_or_magic(w >> 12, magic);
  const f16x2 p0 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, u0) + bias, cs.c_lo, cs.o_lo);
  const f16x2 p1 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, u1) + bias, cs.c_lo, cs.o_lo);
  const f16x2 p2 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, u2) + bias, cs.c_hi, cs.o_hi);
  const f16x2 p3 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, u3) + bias, cs.c_hi, cs.o_hi);
  return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}
__device__ __forceinline__ Q4KF16Consts q4k_f16_consts(i32x4 hdr, int g) {
  const unsigned f = q4k_pair_field((unsigned)hdr[1], (unsigned)hdr[2], (unsigned)hdr[3], g);
  const float d = h2f((unsigned short)((unsigned)hdr[0] & 0xffffu)), dmin = h2f((unsigned short)((unsigned)hdr[0] >> 16));
  const _Float16 c_lo = (_Float16)(d * (float)(f & 63u)), c_hi = (_Float16)(d * (float)((f >> 6) & 63u));  // (11 x 6 bits: exact in f32)
  const _Float16 o_lo = (_Float16)-(dmin * (float)((f >> 12) & 63u)), o_hi = (_Float16)-(dmin * (float)(f >> 18));
  return Q4KF16Consts{f16x2{c_lo, c_lo}, f16x2{o_lo, o_lo}, f16x2{c_hi, c_hi}, f16x2{o_hi, o_hi}};
}

// Q6_K: one dword of ql and the matching dword of qh, already shifted so that bits 0-1 of each byte belong to the low nibbles' quarter
// and bits 4-5 to the high nibbles'
__device__ __forceinline__ unsigned and_or_hi2(unsigned x, unsigned acc) {
  unsigned r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(0x00300030u), "v"(acc));
  return r;
}
__device__ __forceinline__ f16x8 unpack_q6_k_f16(unsigned w, unsigned hw, f16x2 c_lo, f16x2 c_hi, unsigned magic) {
  const f16x2 bias = {(_Float16)-1056.0f, (_Float16)-1056.0f};  // 1024 + q -> q - 32
  const unsigned u0 = and_or_hi2(hw << 4, and_or_magic(w, magic)), u1 = and_or_hi2(hw >> 4, and_or_magic(w >> 8, magic));
  const unsigned u2 = and_or_hi2(hw, and_or_magic(w >> 4, magic)), u3 = and_or_hi2(hw >> 8, and_or_magic(w >> 12, magic));
  const f16x2 p0 = (__builtin_bit_cast(f16x2, u0) + bias) * c_lo, p1 = (__builtin_bit_cast(f16x2, u1) + bias) * c_lo;
  const f16x2 p2 = (__builtin_bit_cast(f16x2, u2) + bias) * c_hi, p3 = (__builtin_bit_cast(f16x2, u3) + bias) * c_hi;
  return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

enum { WF_Q4_0 = 0, WF_Q8_0 = 1, WF_Q4_K = 2, WF_Q6_K = 3, WF_Q4_1 = 4 };  // the weight format of a GEMM

// Up to three weight matrices against the same rhs in ONE launch (wq | wk | wv: the 1024-row k / v GEMMs alone leave most of the
// chip idle for a whole serial k loop): row tile rt belongs to the first matrix whose cumulative tile count exceeds it.
struct F16wMats {
  const i32x4* wq[3];  // the quant plane
  const char* wd[3];   // the scale plane (f16 per block; Q4_1: (d, m); Q4_K: the 16-byte headers; Q6_K: the qh plane)
  const char* ws2[3];  // Q6_K: the int8 scales (16 per super-block) ...
  const char* ws3[3];  // ... and d (f16 per super-block)
  float* out[3];
  float* out2[3];    // ksplit > 1: k piece s >= 1 writes its partial tiles to out2[j] + (s - 1) pstride (k_addn_f32 adds them)
  size_t pstride;
  const unsigned short* exp_tab;  // GU launches: the f16 exp table of silu (silu.rs:6-13)
  F16wHQuant hq;                   // GU launches: h leaves as Q8_0 / Q8_1 planes (+ ffn_down's B') instead of f32 (planes == nullptr: f32)
  int m[3];
  int tiles_end[3];  // cumulative row tiles
};
// h = silu(g) * u (silu.rs:6-13, arithmetic.rs:57-66; fused_ffn.hpp silu_mul: the exp through the reference's f16 table.  Computed instead, the same bits
// for every f16, the launch takes longer: 512 rows of 14336 x 4096 133 -> 139 us.)
__device__ __forceinline__ float f16w_silu_mul(float g, float u, const unsigned short* __restrict__ exp_tab) {
  const float nexp = h2f(exp_tab[f2h(-g)]);
  return (g / (1.0f + nexp)) * u;
}
// h = silu(g) * u of a workgroup's HB 32-row blocks x CW columns, f32 in LDS (H: CS floats a column): ONE THREAD per (column, 32-row block) runs the row
// quantizer on it (quant_lane32's arithmetic, buf_q8_0.rs:87-134 / buf_q8_1.rs:90-129: the block maximum and the integer sum do not depend on the
// order) and writes the block's quants, scale, sum and -- in the slot order of ffn_down's GEMM -- its 32 pre-scaled halfs: h never exists
// as f32 in memory
template <int HB, int CW, int CS, int NT>
__device__ __forceinline__ void f16w_quantize_h(const float* H, const F16wHQuant& hq, int c0, int n, int hb0, int m) {
  const int tid = threadIdx.x;
  const int nbh = m / 32;
  for (int b = tid; b < CW * HB; b += NT) {
    const int col = c0 + b / HB, hb = hb0 + b % HB;
    if (col >= n || hb >= nbh) continue;
    f32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = *(const f32x4*)(H + (b / HB) * CS + 32 * (b % HB) + 4 * j);
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) amax = fmaxf(amax, fabsf(v[j][r]));
    const float dd = amax / 127.0f;
    const unsigned short dh = f2h(dd);
    int q[32], sum = 0;
#pragma unroll
    for (int e = 0; e < 32; e++) {
      const float x = v[e >> 2][e & 3];
      if (hq.q81) {
        q[e] = (int)fminf(fmaxf(x / dd, -128.0f), 127.0f);
      } else {
        q[e] = (int)(signed char)(unsigned char)((unsigned)rs_f32_as_i32(x / dd) & 0xffu);
      }
      sum += q[e];
    }
    char* p = hq.planes + (size_t)col * hq.stride;
    i32x4 pk[2];
#pragma unroll
    for (int e = 0; e < 8; e++)
      pk[e >> 2][e & 3] = (int)(((unsigned)q[4 * e] & 0xffu) | (((unsigned)q[4 * e + 1] & 0xffu) << 8) | (((unsigned)q[4 * e + 2] & 0xffu) << 16) |
                                (((unsigned)q[4 * e + 3] & 0xffu) << 24));
    ((i32x4*)(p + (size_t)hb * 32))[0] = pk[0];
    ((i32x4*)(p + (size_t)hb * 32))[1] = pk[1];
    ((unsigned short*)(p + hq.off_d))[hb] = dh;
    if (hq.q81)
      ((unsigned short*)(p + hq.off_aux))[hb] = f2h((float)sum * dd);
    else
      ((int*)(p + hq.off_aux))[hb] = sum;
    if (hq.xh != nullptr) {
      const float ds = h2f(dh);
      unsigned short* xr = hq.xh + ((size_t)col * nbh + hb) * 32;
#pragma unroll
      for (int s4 = 0; s4 < 4; s4++) {
        unsigned short o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = f16w_value(q[f16w_slot_elem(8 * s4 + e)], ds);
        *(i32x4*)(xr + 8 * s4) = i32x4{(int)(o[0] | ((unsigned)o[1] << 16)), (int)(o[2] | ((unsigned)o[3] << 16)),
                                       (int)(o[4] | ((unsigned)o[5] << 16)), (int)(o[6] | ((unsigned)o[7] << 16))};
      }
    }
  }
}

// what a chunk of k takes a launch over its rounds of CUs, where a workgroup's takes `alone` with a CU to itself and `shared` beside another (0: it has one to itself)
inline float f16w_chunk_us(size_t wgs, size_t n_cu, float alone, float shared, float* rounds) {
  const size_t slots = n_cu * (shared > 0.f ? 2 : 1), rest = wgs % slots;
  *rounds = (float)(wgs / slots) + (rest != 0);
  return (float)(wgs / slots) * (shared > 0.f ? shared : alone) + (rest == 0 ? 0.f : rest <= n_cu ? alone : shared);
}
// gemm_f16w_wide.hip, passes of more than 64 rows, k a multiple of 256.  Estimated time of the launch that it would make, us; deferred: pieces of k are the consumer's
float f16w_wide_us(uint32_t dt, const size_t* m, int nw, size_t k, size_t b, size_t n_cu, size_t ws_floats, bool deferred);
// false: not covered.  ksplit: the pieces of k that a launch of its own or the consumer adds
bool launch_f16w_wide(crabml_hip_device* dev, uint32_t dt, F16wMats mats, const size_t* m, int nw, size_t k, const void* xh, size_t b, bool pair, bool gu,
                      size_t ws_floats, int* ksplit);

}  // namespace crabml_hip
