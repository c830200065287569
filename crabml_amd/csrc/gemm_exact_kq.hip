// gemm_exact_kq.hip -- Q4_K weights x several Q8_K rows in the reference's order (the strict device's prompts), on the int8 matrix cores
//
// buf_q4_k.rs:192-277 keeps eight f32 lanes per output: sums[l] += d * A[l] super-block after super-block, with A[l] the exact integer sum of
// scale * q4 * q8 over the elements e with e % 8 == l, beside sumf -= dmin * sumi; the lanes are added at the end, in order.  The nine chains do not
// depend on each other, so a workgroup owns a tile of outputs and each of its nine waves runs one chain over all super-blocks; the waves meet once.
//   A[l]: a class has 4 elements of each of the 8 sub-blocks, 32 in all -- one v_mfma_i32_16x16x32_i8 -- and with the planes class-major (common.hpp) lane
//   (i, g) finds its 8 bytes in dword l of chunk g: low nibbles of sub-block 2 g, high nibbles of 2 g + 1.  The 6-bit scale goes into the weights' bytes in
//   two halves of 3 bits (15 * 7 < 128): A[l] = 8 * (scale >> 3 part) + (scale & 7 part), in integers.
//   sumi: the 6-bit minimums against the sub-blocks' sums of quants as 64 a + b, both of them bytes.
// D's rows are rows of the rhs, its columns rows of the matrix, so that d is the lane's own.  Reads, products and sums are k_gemv_exact_q4k's values in
// its order: the same bits.  What bounds it is vector work: some 40 instructions a wave, super-block and tile of the rhs, half of them the reference's f32
// terms.  11 rows, us a launch, row kernels / this: 14336 x 4096 69.8 / 27.6, 4096 x 4096 and 4096 x 14336 39.5 / 14.1 on average, 1024 x 4096 9.3 / 9.0.
#include <type_traits>

#include "common.hpp"
#include "devutil.hpp"
#include "gemv_core.hpp"
#include "kernels.hpp"

namespace crabml_hip {

#define KQX_WAVES 9
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

struct KqxArgs {
  const char *w, *wh;  // qs | hdr planes
  const char* act;
  size_t act_stride, off_d, off_aux, off_p;
  float* out;        // [b][m]
  const float* add;  // [b][m] (nullable; may be out)
  int m, nsb, b, row_tiles, col_tiles;
};

// the four bytes of q times s (<= 7; bytes <= 15)
__device__ __forceinline__ unsigned kqx_scaled(unsigned q, unsigned s) {
  return __builtin_bit_cast(unsigned, (u16x2)(__builtin_bit_cast(u16x2, q) * (u16x2){(unsigned short)s, (unsigned short)s}));
}
__device__ __forceinline__ long kqx_pair(unsigned lo, unsigned hi) { return (long)(((unsigned long long)hi << 32) | lo); }

// NT: 16-row tiles of the rhs per workgroup.  Super-blocks go through LDS a stage of G at a time, laid out as the lanes of a class read them: a lane's dword
// straight from memory is 16 lines a request, nine times over (14336 x 4096, 11 rows: 76 to 106 us, through LDS 27.6).
template <int NT>
struct KqxTile {
  static constexpr int G = NT == 1 ? 4 : 2, CW = 16 * NT, PS = 72;  // PS: dwords of a class of 16 rows' chunks, so that a 16-byte piece's two halves meet other banks
  // one stage, in dwords per super-block: weights [8][PS], their fields [16][4] and d | dmin [16]; the rhs [8][NT][16][4][2], sums of 16 quants [NT][16][4][2], d [CW]
  static constexpr int O_F = 8 * PS, O_H = O_F + 64, O_X = O_H + 16, O_S = O_X + 8 * NT * 128, O_D = O_S + NT * 128, SB = O_D + CW;
  static constexpr int OS = 17, ENDS = KQX_WAVES * CW * OS;  // the chains' ends [9][CW][OS]
  static constexpr int LDS = 2 * G * SB > ENDS ? 2 * G * SB : ENDS;
  static constexpr int XP = G * NT / 2, AP = G / 4 > 0 ? G / 4 : 1;  // 16-byte pieces of a thread: rhs, weights (G = 2: of every second thread)
};

template <int NT>
__global__ __launch_bounds__(64 * KQX_WAVES) void k_gemm_exact_q4k(const KqxArgs a) {
  using T = KqxTile<NT>;
  constexpr int CW = T::CW, G = T::G;
  extern __shared__ __attribute__((aligned(16))) unsigned kqx_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg(), i = lane & 15, g = lane >> 4;
  int rt, ct;
  if ((a.row_tiles & 7) == 0) {  // a row tile's workgroups back to back on one XCD
    const int x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
    ct = j % a.col_tiles;
    rt = j / a.col_tiles * 8 + x;
  } else {
    rt = (int)blockIdx.x % a.row_tiles;
    ct = (int)blockIdx.x / a.row_tiles;
  }
  const int r0 = rt * 16, c0 = ct * CW, nsb = a.nsb, stages = (nsb + G - 1) / G;
  auto row_of = [&](int r) { return r0 + r < a.m ? r0 + r : a.m - 1; };
  auto col_of = [&](int c) { return c0 + c < a.b ? c0 + c : a.b - 1; };
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // D += over a stage: f the lane's two sub-blocks' fields, h its row's d and dmin
  auto terms = [&](auto mins, const unsigned* S) {
    constexpr bool MINS = decltype(mins)::value;
    const unsigned f = S[T::O_F + i * 4 + g], h = S[T::O_H + i], q = MINS ? 0u : S[wave * T::PS + i * 4 + g];
    const i32x4 zero = {0, 0, 0, 0};
    const float d = h2f((unsigned short)(MINS ? h >> 16 : h & 0xffffu));
    const unsigned lo = q & 0x0F0F0F0Fu, hi = (q >> 4) & 0x0F0F0F0Fu;
    const long w1 = MINS ? (long)(((f >> 12) & 63u) | (f >> 18) << 8) : kqx_pair(kqx_scaled(lo, (f >> 3) & 7u), kqx_scaled(hi, (f >> 9) & 7u));
    const long w0 = MINS ? w1 : kqx_pair(kqx_scaled(lo, f & 7u), kqx_scaled(hi, (f >> 6) & 7u));
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const u32x2 x = *(const u32x2*)(S + (MINS ? T::O_S : T::O_X + wave * NT * 128) + t * 128 + (i * 4 + g) * 2);
      long x1 = kqx_pair(x[0], x[1]), x0 = x1;
      if constexpr (MINS) {
        const int s_lo = (int)(short)(x[0] & 0xffffu) + ((int)x[0] >> 16), s_hi = (int)(short)(x[1] & 0xffffu) + ((int)x[1] >> 16);
        const int a_lo = (s_lo + 32) >> 6, a_hi = (s_hi + 32) >> 6;  // |sum| <= 32 * 128: a in [-64, 64], b in [-32, 32)
        x1 = (long)((a_lo & 255) | (a_hi & 255) << 8);
        x0 = (long)(((s_lo - 64 * a_lo) & 255) | ((s_hi - 64 * a_hi) & 255) << 8);
      }
      const i32x4 p1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(x1, w1, zero, 0, 0, 0), p0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(x0, w0, zero, 0, 0, 0);
      const i32x4 p = (p1 << (MINS ? 6 : 3)) + p0;
      const f32x4 d8 = *(const f32x4*)(S + T::O_D + t * 16 + g * 4);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float v = (d * d8[e]) * (float)p[e];
        acc[t][e] = MINS ? acc[t][e] - v : acc[t][e] + v;
      }
    }
  };
  // (stages end in super-blocks past the last one: they read it again, and are not added)
  auto chain = [&](auto mins, auto&& fetch, auto&& commit) {
    fetch(0);
    commit(kqx_lds);
    fetch(1);
    __syncthreads();
    for (int s = 0; s < stages; s++) {
      const unsigned* S = kqx_lds + (s & 1) * G * T::SB;
      if ((s + 1) * G <= nsb) {
#pragma unroll
        for (int u = 0; u < G; u++) terms(mins, S + u * T::SB);
      } else {
        for (int u = 0; s * G + u < nsb; u++) terms(mins, S + u * T::SB);
      }
      commit(kqx_lds + ((s + 1) & 1) * G * T::SB);
      fetch(s + 2);
      __syncthreads();
    }
  };
  if (wave < 8) {  // the classes; between them the weights' quants and the rhs
    i32x4 ra[T::AP], rx[T::XP];
    const char* wp;
    const char* xp[T::XP];
    int wu, wat, xu[T::XP], xat[T::XP];
    {
      const int p = tid % (128 * G), r = p & 127, row = r >> 3, pc = r & 7;  // piece pc: half pc & 1 of chunk pc / 2
      wu = p >> 7;
      wp = a.w + (size_t)row_of(row) * nsb * 128 + pc * 16;
      wat = wu * T::SB + (pc & 1) * 4 * T::PS + row * 4 + (pc >> 1);
    }
#pragma unroll
    for (int v = 0; v < T::XP; v++) {
      const int p = tid + v * 512, r = p % (256 * NT), col = r >> 4, pc = r & 15;  // pair pc / 4, low or high nibbles' elements, half
      xu[v] = p / (256 * NT);
      xp[v] = a.act + (size_t)col_of(col) * a.act_stride + a.off_p + pc * 16;
      xat[v] = xu[v] * T::SB + T::O_X + (pc & 1) * 4 * NT * 128 + (col >> 4) * 128 + ((col & 15) * 4 + (pc >> 2)) * 2 + ((pc >> 1) & 1);
    }
    auto fetch = [&](int s) {
      const int w = s * G + wu < nsb ? s * G + wu : nsb - 1;
      ra[0] = *(const i32x4*)(wp + (size_t)w * 128);
#pragma unroll
      for (int v = 0; v < T::XP; v++) {
        const int x = s * G + xu[v] < nsb ? s * G + xu[v] : nsb - 1;
        rx[v] = *(const i32x4*)(xp[v] + (size_t)x * 256);
      }
    };
    auto commit = [&](unsigned* S) {
      if (tid < 128 * G) {
#pragma unroll
        for (int e = 0; e < 4; e++) S[wat + e * T::PS] = (unsigned)ra[0][e];
      }
#pragma unroll
      for (int v = 0; v < T::XP; v++)
#pragma unroll
        for (int e = 0; e < 4; e++) S[xat[v] + e * NT * 128] = (unsigned)rx[v][e];
    };
    chain(std::false_type{}, fetch, commit);
  } else {  // the minimums; the weights' headers, the rhs rows' sums and d
    unsigned rf[G], rh[G];
    u32x2 rs[G][NT];
    float rd[G * NT / 4 > 0 ? G * NT / 4 : 1];
    const char* wh = a.wh + (size_t)row_of(i) * nsb * 16;
    const char* xs[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) xs[t] = a.act + (size_t)col_of(t * 16 + i) * a.act_stride;
    auto fetch = [&](int s) {
#pragma unroll
      for (int u = 0; u < G; u++) {
        const int sb = s * G + u < nsb ? s * G + u : nsb - 1;
        rh[u] = *(const unsigned*)(wh + (size_t)sb * 16);
        __builtin_memcpy(&rf[u], wh + (size_t)sb * 16 + 3 + 3 * g, 4);  // the pair's 24-bit field in the upper bytes
#pragma unroll
        for (int t = 0; t < NT; t++) rs[u][t] = *(const u32x2*)(xs[t] + a.off_aux + (size_t)sb * 32 + g * 8);
      }
#pragma unroll
      for (int v = 0; v < (int)(sizeof rd / 4); v++) {  // lane (i, g): column block and super-block v * 4 + g
        const int e = v * 4 + g < G * NT ? v * 4 + g : 0, t = e % NT, sb = s * G + e / NT < nsb ? s * G + e / NT : nsb - 1;
        rd[v] = *(const float*)(a.act + (size_t)col_of(t * 16 + i) * a.act_stride + a.off_d + (size_t)sb * 4);
      }
    };
    auto commit = [&](unsigned* S) {
#pragma unroll
      for (int u = 0; u < G; u++) {
        S[u * T::SB + T::O_F + i * 4 + g] = rf[u] >> 8;
        if (g == 0) S[u * T::SB + T::O_H + i] = rh[u];
#pragma unroll
        for (int t = 0; t < NT; t++) *(u32x2*)(S + u * T::SB + T::O_S + t * 128 + (i * 4 + g) * 2) = rs[u][t];
      }
#pragma unroll
      for (int v = 0; v < (int)(sizeof rd / 4); v++) {
        const int e = v * 4 + g;
        if (e < G * NT) S[e / NT * T::SB + T::O_D + e % NT * 16 + i] = __builtin_bit_cast(unsigned, rd[v]);
      }
    };
    chain(std::true_type{}, fetch, commit);
  }
  float* ends = (float*)kqx_lds;
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int e = 0; e < 4; e++) ends[(wave * CW + t * 16 + g * 4 + e) * T::OS + i] = acc[t][e];
  __syncthreads();
  for (int e = tid; e < CW * 16; e += 64 * KQX_WAVES) {
    const int c = e >> 4, r = e & 15;
    if (c0 + c >= a.b || r0 + r >= a.m) continue;
    float s = ends[(8 * CW + c) * T::OS + r];
#pragma unroll
    for (int l = 0; l < 8; l++) s += ends[(l * CW + c) * T::OS + r];
    const size_t at = (size_t)(c0 + c) * a.m + r0 + r;
    a.out[at] = a.add ? s + a.add[at] : s;
  }
}

template <int NT>
static bool launch_t(crabml_hip_device* dev, const KqxArgs& a) {
  const size_t lds = (size_t)KqxTile<NT>::LDS * 4;
  if (raise_dyn_lds(dev, (const void*)k_gemm_exact_q4k<NT>, (int)lds) != hipSuccess) return false;
  launch_k(dev->stream, nullptr, k_gemm_exact_q4k<NT>, dim3(a.row_tiles * a.col_tiles), dim3(64 * KQX_WAVES), lds, a);
  return true;
}

// false: not covered (the caller's row kernels take it)
bool launch_gemm_exact_kq(crabml_hip_device* dev, const crabml_hip_buf* w, size_t m, size_t k, const void* act, size_t b, float* out, const float* add) {
  const int nsb = (int)(k / 256);
  // tiles of 16 rows a workgroup: a workgroup of one, two and four costs as 26 : 50 : 81 (a prompt on four layers of the 8B shape, us: 77 rows 1753 / 1979 / 2146, 64 rows
  // 1558 / 1442 / 1401, 100 rows 2320 / 2437 / 2170, 17 rows 995 / 1015 / 1399), empty tiles included
  const size_t tiles = (b + 15) / 16;
  int nt = 1;
  size_t least = tiles * 26;
  for (int n : {2, 4}) {
    const size_t cost = (tiles + n - 1) / n * (n == 2 ? 50 : 81);
    if (cost < least) {
      least = cost;
      nt = n;
    }
  }
  if (w->dtype != CRABML_HIP_Q4_K || b < KQX_ROWS || m == 0 || nsb == 0) return false;
  const ActLayout al = act_layout(CRABML_HIP_Q8_K, k);
  KqxArgs a;
  a.w = (const char*)w->ptr;
  a.wh = a.w + w->wl.off_scale;
  a.act = (const char*)act;
  a.act_stride = al.total;
  a.off_d = al.off_d;
  a.off_aux = al.off_aux;
  a.off_p = al.off_p;
  a.out = out;
  a.add = add;
  a.m = (int)m;
  a.nsb = nsb;
  a.b = (int)b;
  a.row_tiles = (int)((m + 15) / 16);
  a.col_tiles = (int)((b + 16 * nt - 1) / (16 * nt));
  if ((size_t)a.row_tiles * a.col_tiles > 0x7fffffffu / (64 * KQX_WAVES)) return false;
  return nt == 1 ? launch_t<1>(dev, a) : nt == 2 ? launch_t<2>(dev, a) : launch_t<4>(dev, a);
}

}  // namespace crabml_hip
