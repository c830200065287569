// devutil.hpp -- small device helpers shared by the kernels (gfx950: wave = 64 lanes).
#pragma once
#include "common.hpp"

namespace crabml_hip {

// A pointer that a kernel reads from memory (a sequence's slab) is generic to the compiler, and generic loads count as LDS accesses too:
// every wait for LDS then waits for them.  This says that it points to device memory.
template <typename T>
__device__ __forceinline__ T* as_global(T* p) {
  return (T*)(__attribute__((address_space(1))) T*)(size_t)p;
}

// half crate semantics: from_f32 = IEEE RNE (v_cvt_f16_f32 in the default round mode), to_f32 exact.
__device__ __forceinline__ float h2f(unsigned short h) {
  _Float16 x;
  __builtin_memcpy(&x, &h, 2);
  return (float)x;
}
__device__ __forceinline__ unsigned short f2h(float f) {
  // The empty asm pins the f32 value in a VGPR first.  Without it hipcc folds f16(a*b) / f16(a+b) into
  // v_fma_mixlo_f16 (a*b + 0 rounded ONCE to f16): that drops the sign of a -0.0 product and skips the
  // intermediate f32 rounding the half crate performs -- seen on MI355X as Q8_1 `s` = +0 instead of -0.
  asm("" : "+v"(f));  // (not volatile: may be scheduled freely, only the value is opaque)
  _Float16 x = (_Float16)f;
  unsigned short h;
  __builtin_memcpy(&h, &x, 2);
  return h;
}
// eight f16 x f16 products, exact in f32, added to s one after the other
__device__ __forceinline__ float dot_f16x8(i32x4 a, i32x4 b, float s) {
  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  const h8 x = __builtin_bit_cast(h8, a), y = __builtin_bit_cast(h8, b);
#pragma unroll
  for (int e = 0; e < 8; e++) s = __builtin_fmaf((float)x[e], (float)y[e], s);
  return s;
}
// bfloat16: the upper half of an f32 (exact), and back with round-to-nearest-even
__device__ __forceinline__ float bf2f(unsigned short h) { return __builtin_bit_cast(float, (unsigned)h << 16); }
__device__ __forceinline__ unsigned short f2bf(float f) {
  const __bf16 x = (__bf16)f;
  return __builtin_bit_cast(unsigned short, x);
}
// half: `a * b` / `a + b` on f16 = compute in f32, round once to f16
__device__ __forceinline__ unsigned short h_mul(unsigned short a, unsigned short b) { return f2h(h2f(a) * h2f(b)); }
__device__ __forceinline__ unsigned short h_add(unsigned short a, unsigned short b) { return f2h(h2f(a) + h2f(b)); }

// Native f16 arithmetic.  The half crate computes `a * b` / `a + b` in f32 and rounds once to f16; for + and * that
// double rounding is innocuous (24 >= 2 * 11 + 2 significand bits), so it equals ONE correctly rounded f16
// operation: v_mul_f16 / v_add_f16.  Used by the f16-accumulated PV chain of attention (buf_f16.rs:152-163), where
// the add is a serial dependency per cached position (1 dependent instruction instead of 3).  Compiled with
// -ffp-contract=off: the product and the sum stay two roundings.
__device__ __forceinline__ _Float16 hbits(unsigned short h) {
  _Float16 x;
  __builtin_memcpy(&x, &h, 2);
  return x;
}
__device__ __forceinline__ unsigned short hraw(_Float16 x) {
  unsigned short h;
  __builtin_memcpy(&h, &x, 2);
  return h;
}

// ---- cross-lane reductions on DPP (gfx9 data-parallel primitives) -------------------------------------
// __shfl_xor lowers to ds_bpermute_b32 (an LDS-crossbar round trip, ~100 cycles each, and a 5-6 deep
// dependent chain per reduction); measured on MI355X this made the single-workgroup norm+quantize stage
// 13.8 us.  DPP row operations are register-to-register: 4 steps reduce each 16-lane row, v_readlane
// combines the 4 rows.  All lanes must be active (callers keep whole waves converged).
// the wave's index inside its workgroup as a SCALAR (threadIdx.x >> 6 is uniform per wave, but the compiler cannot know: everything
// derived from it -- the rows a wave owns, their base addresses -- then lives in VGPRs and every address is 64-bit vector arithmetic;
// through readfirstlane the row bases become SGPR pairs and the loads take the `saddr + 32-bit lane offset` form)
__device__ __forceinline__ int wave_in_wg() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, dpp_i<CTRL>(__builtin_bit_cast(int, v)));
}
// DPP controls: quad_perm[1,0,3,2]=0xB1, quad_perm[2,3,0,1]=0x4E, row_half_mirror=0x141, row_mirror=0x140
__device__ __forceinline__ float row16_sum_f32(float v) {
  v += dpp_f<0xB1>(v);
  v += dpp_f<0x4E>(v);
  v += dpp_f<0x141>(v);
  v += dpp_f<0x140>(v);
  return v;
}
__device__ __forceinline__ float row16_max_f32(float v) {
  v = fmaxf(v, dpp_f<0xB1>(v));
  v = fmaxf(v, dpp_f<0x4E>(v));
  v = fmaxf(v, dpp_f<0x141>(v));
  v = fmaxf(v, dpp_f<0x140>(v));
  return v;
}
__device__ __forceinline__ int row16_sum_i32(int v) {
  v += dpp_i<0xB1>(v);
  v += dpp_i<0x4E>(v);
  v += dpp_i<0x141>(v);
  v += dpp_i<0x140>(v);
  return v;
}
__device__ __forceinline__ float rl_f(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
// half waves / neighbouring rows of 16 lanes swap and add: the first half (even rows) gets a's sum, the other half (odd rows) b's
__device__ __forceinline__ float meet32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned lo = r[0], hi = r[1];
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ float meet16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned lo = r[0], hi = r[1];
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
// the larger of the two, in both
__device__ __forceinline__ float max32(float a) {
  const unsigned u = __builtin_bit_cast(unsigned, a);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const unsigned lo = r[0], hi = r[1];
  return fmaxf(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi));
}
__device__ __forceinline__ float max16(float a) {
  const unsigned u = __builtin_bit_cast(unsigned, a);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned lo = r[0], hi = r[1];
  return fmaxf(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi));
}
// Sums over the 64 / LPR groups of LPR lanes.  Of a lane's eight columns it is left with the sums of two -- pair 2 (lane / 32) + (lane / 16) % 2
// of the four -- in acc[0], acc[1] (LPR = 32: of four, half lane / 32 of the eight).  LPR = 8: lanes 8-15 of a row hold what lanes 0-7 do.
template <int LPR>
__device__ __forceinline__ void sum_groups(float (&acc)[8]) {
#pragma unroll
  for (int i = 0; i < 4; i++) acc[i] = meet32(acc[i], acc[i + 4]);
  if constexpr (LPR < 32) {
    acc[0] = meet16(acc[0], acc[2]);
    acc[1] = meet16(acc[1], acc[3]);
  }
  if constexpr (LPR == 8) {
    acc[0] += dpp_f<0x128>(acc[0]);
    acc[1] += dpp_f<0x128>(acc[1]);
  }
}
template <int LPR>
__device__ __forceinline__ float sum_groups(float v) {
  v = meet32(v, v);
  if constexpr (LPR < 32) v = meet16(v, v);
  if constexpr (LPR == 8) v += dpp_f<0x128>(v);
  return v;
}
// the sum over a group's lanes, in all of them
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
  v += dpp_f<0xB1>(v);
  v += dpp_f<0x4E>(v);
  v += dpp_f<0x141>(v);
  if constexpr (LPR >= 16) v += dpp_f<0x140>(v);
  if constexpr (LPR == 32) v = meet16(v, v);
  return v;
}
// full-wave (64 lanes): every lane gets the result
__device__ __forceinline__ float wave_sum_f32(float v) {
  v = row16_sum_f32(v);
  return (rl_f(v, 0) + rl_f(v, 16)) + (rl_f(v, 32) + rl_f(v, 48));
}
__device__ __forceinline__ float wave_max_f32(float v) {
  v = row16_max_f32(v);
  return fmaxf(fmaxf(rl_f(v, 0), rl_f(v, 16)), fmaxf(rl_f(v, 32), rl_f(v, 48)));
}
// per 32-lane half (one Q8_0 block per half-wave): lanes 0-31 get their half's result, lanes 32-63 theirs
__device__ __forceinline__ float half_max_f32(float v) {
  v = row16_max_f32(v);
  float lo = fmaxf(rl_f(v, 0), rl_f(v, 16)), hi = fmaxf(rl_f(v, 32), rl_f(v, 48));
  return (threadIdx.x & 32) ? hi : lo;
}
__device__ __forceinline__ int half_sum_i32(int v) {
  v = row16_sum_i32(v);
  int lo = __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16);
  int hi = __builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48);
  return (threadIdx.x & 32) ? hi : lo;
}

// Q4_K header words u0..u2 (the re-packed scales, common.hpp) -> the 24-bit field of pair p:
// scale[2p] | scale[2p+1] << 6 | min[2p] << 12 | min[2p+1] << 18
__device__ __forceinline__ unsigned q4k_pair_field(unsigned u0, unsigned u1, unsigned u2, int p) {
  const unsigned lo = p == 0 ? u0 : p == 1 ? u0 : p == 2 ? u1 : u2;
  const unsigned hi = p == 0 ? u0 : p == 1 ? u1 : p == 2 ? u2 : u2;
  const unsigned sh = p == 0 ? 0u : p == 1 ? 24u : p == 2 ? 16u : 8u;
  return (unsigned)(((((unsigned long long)hi) << 32) | lo) >> sh) & 0xffffffu;
}

// Rust `f32 as i32`: saturating, NaN -> 0
__device__ __forceinline__ int rs_f32_as_i32(float v) {
  if (v != v) return 0;
  if (v >= 2147483648.0f) return 2147483647;
  if (v <= -2147483648.0f) return (-2147483647 - 1);
  return (int)v;
}

template <bool NT, typename T>
__device__ __forceinline__ T ld(const T* p) {
  if constexpr (NT)
    return __builtin_nontemporal_load(p);
  else
    return *p;
}

// Q8_0 / Q8_1 quantizer of 32-element blocks, 8 lanes of 4 consecutive elements each (buf_q8_0.rs:87-134, buf_q8_1.rs:90-129; quant_lane32's arithmetic,
// fused_common.hpp: the maximum and the integer sum do not depend on the order).  aux: the sum of the quants, or Q8_1's s as f16 bits; all lanes of the block get d and aux.
struct QLane4 {
  unsigned packed;
  unsigned short d;
  int aux;
};
template <bool Q81>
__device__ __forceinline__ QLane4 quant_quad8(const f32x4 v) {
  float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
  amax = fmaxf(amax, dpp_f<0xB1>(amax));
  amax = fmaxf(amax, dpp_f<0x4E>(amax));
  amax = fmaxf(amax, dpp_f<0x141>(amax));
  const float dd = amax / 127.0f;
  QLane4 o;
  o.d = f2h(dd);
  int q[4], s = 0;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    if constexpr (Q81)
      q[e] = (int)fminf(fmaxf(v[e] / dd, -128.0f), 127.0f);  // Rust f32::max / min return the non-NaN operand
    else
      q[e] = (int)(signed char)(unsigned char)((unsigned)rs_f32_as_i32(v[e] / dd) & 0xffu);  // `as i8` from i32 wraps
    s += q[e];
  }
  s += dpp_i<0xB1>(s);
  s += dpp_i<0x4E>(s);
  s += dpp_i<0x141>(s);
  o.aux = Q81 ? (int)f2h((float)s * dd) : s;
  o.packed = ((unsigned)q[0] & 0xffu) | (((unsigned)q[1] & 0xffu) << 8) | (((unsigned)q[2] & 0xffu) << 16) | ((unsigned)q[3] << 24);
  return o;
}

// Q8_K quantizer of one 256-element super-block by one wave, 4 consecutive elements per lane
// (buf_q8_k.rs:84-131: scale = -128 / (the FIRST element of maximal |x|), round half away from zero, min(127),
// `as i8` saturation).  Returns the 4 quants packed into a dword; `quad_sum` = this lane's quad's sum of 16 quants
// (bsums entry lane/4), `d` = the block scale (0 for an all-zero block).
struct Q8KLane {
  unsigned packed;
  int quad_sum;
  float d;
};
__device__ __forceinline__ Q8KLane q8k_wave_quant(const f32x4 v, int lane) {
  // first element of maximal |x| -- of its value only the sign is not known yet: the wave maximum by DPP, the lowest lane that holds it (ballot), that
  // lane's first element that does.  (NaN is never the maximum.)
  const float best_abs = wave_max_f32(fmaxf(fmaxf(fmaxf(0.f, fabsf(v[0])), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
  float mine = 0.f;
#pragma unroll
  for (int i = 3; i >= 0; i--) mine = fabsf(v[i]) == best_abs ? v[i] : mine;
  const unsigned long long holders = __ballot(fabsf(mine) == best_abs);
  const float best_val = rl_f(mine, holders ? __builtin_ctzll(holders) : 0);
  const float scale = -128.0f / best_val;
  Q8KLane o;
  o.d = best_abs == 0.0f ? 0.0f : 1.0f / scale;
  int qi[4];
  int s = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    // half away from zero: the largest number below 1/2 moves exactly what rounds up past the next integer (every |r| to 131), the conversion cuts off.
    // min(127) takes NaN to 127, `as i8` saturates.
    float r = scale * v[i];
    r = fmaxf(fminf(r + __builtin_copysignf(0.49999997f, r), 127.0f), -128.0f);
    const int t = best_abs != 0.0f ? (int)r : 0;
    qi[i] = t;
    s += t;
  }
  o.packed = ((unsigned)qi[0] & 0xffu) | (((unsigned)qi[1] & 0xffu) << 8) | (((unsigned)qi[2] & 0xffu) << 16) | ((unsigned)qi[3] << 24);
  s += dpp_i<0xB1>(s);
  s += dpp_i<0x4E>(s);
  o.quad_sum = s;
  return o;
}

// The class-major copy of a super-block's quants (plane `qp`, common.hpp): q8k_wave_quant leaves lane L the four consecutive
// elements 4 L .. 4 L + 3; element 4 j + k of 32-group c = L / 8 (j = L % 8) goes to byte 4 ((4 j + k) % 8) + (4 j + k) / 8 =
// 16 (j & 1) + 4 k + j / 2 of the group: four bytes of four lanes of one parity are transposed (two exchanges), after which a lane holds dword
// 4 (j & 1) + j / 2 of its group.  sb_base: the super-block's 256 bytes (global memory or LDS), 4-byte aligned.  All lanes of the wave.
__device__ __forceinline__ unsigned q8k_class_major(int lane, unsigned packed) {
  const unsigned a = (unsigned)dpp_i<0x4E>((int)packed);  // of lane ^ 2
  packed = __builtin_amdgcn_perm(a, packed, lane & 2 ? 0x03070105u : 0x06020400u);
  const unsigned b = (unsigned)dpp_i<0x1B>(dpp_i<0x141>((int)packed));  // of lane ^ 4 (half row mirrored, quads mirrored)
  return __builtin_amdgcn_perm(b, packed, lane & 4 ? 0x03020706u : 0x05040100u);
}
__device__ __forceinline__ int q8k_class_major_at(int lane) { return (lane >> 3) * 8 + (lane & 1) * 4 + ((lane >> 1) & 3); }
// (`in`: lanes that store, each a whole dword of its own)
__device__ __forceinline__ void q8k_store_class_major(signed char* sb_base, int lane, unsigned packed, bool in = true) {
  const unsigned d = q8k_class_major(lane, packed);
  if (in) ((unsigned*)sb_base)[q8k_class_major_at(lane)] = d;
}

}  // namespace crabml_hip
