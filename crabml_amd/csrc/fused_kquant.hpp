// fused_kquant.hpp -- the fast decode step over Q4_K and Q6_K weights: every launch makes the Q8_K planes of its rhs itself, in LDS, from an f32 row.
//
// Per layer: [norm + quantize + q | k | v + rope + append], attention, [quantize + wo + residual], [norm + quantize + gate | up + SiLU * mul], [quantize +
// ffn_down + residual].  A Q8_K super-block is 256 elements whose scale comes from the first one of maximal |x|, and the producers own 16 or 32 rows each:
// a producer that leaves planes has to meet its neighbours inside its launch (granules, 2.4 us behind gate | up of 14336 rows; with the norm's
// sum of squares 2.7 behind ffn_down), with nothing on its way meanwhile.  A consumer's own quantizer runs under its first weight requests: it is a
// wave per super-block and some 60 instructions (q8k_wave_quant).  Bound: the weights' bytes, plus a launch's ramp.
// Every row's pieces are added by lane, ascending, as k_gemv_q4_k / k_gemv_q6_k add them, the norm's sums in k_norm_f32's order: the planes and logits are the per-op
// launches' bit for bit.
// Us a launch of the 8B shape, Q4_K, with planes from the producer / these: q | k | v 5.6 / 5.8, wo 5.6 / 4.4, gate | up 16.6 / 13.7 (4.8 TB/s), ffn_down 11.2 / 9.0; on the
// strict-order device (ORD) 7.2 / 9.6, 11.3 / 5.6, 19.8 / 18.7, 16.8 / 12.4 (in a kernel trace).  A token of four layers 269 -> 242, of Q6_K (fourteen launches a layer and the attention before)
// 407 -> 297; width 2048, six layers, Q4_K 222 -> 192, Q6_K 363 -> 214.
#pragma once
#include "fused_ffn.hpp"

namespace crabml_hip {

// a matrix: Q4_K planes qs | headers at off, Q6_K planes ql | qh at off | scales | d
struct KqMat {
  const char* p;
  size_t off;
};

// one lane's piece c of a row: 16 bytes of quants with what goes with them, and its share of the rhs
template <bool SIX>
struct KqPiece;
template <>
struct KqPiece<false> {
  Q4KPiece<false> w;
};
template <>
struct KqPiece<true> {
  i32x4 ql, qh;
  i32x2 sc;  // scales of the eight groups of the piece's half, those of gi and gi + 4 among them
  unsigned short d;
};
// (row: the same for the whole wave -- the row's planes are scalar addresses, a lane adds 32 bits)
template <bool SIX>
__device__ __forceinline__ KqPiece<SIX> kq_load(const KqMat& m, int row, int nsb, int c) {
  KqPiece<SIX> p;
  const size_t blk0 = (size_t)row * nsb;
  const unsigned u = (unsigned)c, sb = u >> 3;
  auto at = [&](const char* base, unsigned off) { return as_global(base) + off; };
  if constexpr (!SIX) {
    p.w.qv = __builtin_nontemporal_load((const i32x4*)at(m.p + blk0 * 128, u * 16));
    p.w.hdr = __builtin_nontemporal_load((const i32x4*)at(m.p + m.off + blk0 * 16, sb * 16));
  } else {
    const size_t n = m.off / 128;
    p.ql = __builtin_nontemporal_load((const i32x4*)at(m.p + blk0 * 128, u * 16));
    p.qh = __builtin_nontemporal_load((const i32x4*)at(m.p + m.off + blk0 * 64, sb * 64 + ((u >> 1) & 2) * 16 + (u & 1) * 16));  // (rows_partial_q6k)
    p.sc = *(const i32x2*)at(m.p + m.off + n * 64 + blk0 * 16, sb * 16 + ((u >> 2) & 1) * 8);
    p.d = *(const unsigned short*)at(m.p + m.off + n * 80 + blk0 * 2, sb * 2);
  }
  return p;
}
template <bool SIX>
__device__ __forceinline__ Q4KX kq_loadx(const ActQ8_K& act, int c) {
  if constexpr (!SIX) return q4k_loadx(act, c);
  const int sb = c >> 3, gi = 8 * ((c >> 2) & 1) + (c & 1) + 2 * ((c >> 1) & 1);
  Q4KX x;
  const i32x4* xq = act.q + (size_t)sb * 16 + gi;  // 16 int8 a group
  x.xl = xq[0];
  x.xh = xq[4];
  x.d8 = act.d[sb];
  const short* bs = act.bsums + sb * 16 + gi;
  x.bs_lo = (int)bs[0];
  x.bs_hi = (int)bs[4];
  return x;
}
template <bool SIX>
__device__ __forceinline__ float kq_term(const KqPiece<SIX>& p, const Q4KX& x, int c) {
  if constexpr (!SIX) {
    return q4k_term<false>(p.w, x, c);
  } else {
    const int a = (c >> 1) & 1;
    int lo = 0, hi = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const unsigned q = (unsigned)p.ql[i], hb = (unsigned)p.qh[i] >> (2 * a);
      lo = __builtin_amdgcn_sdot4((int)((q & 0x0F0F0F0Fu) | ((hb & 0x03030303u) << 4)), x.xl[i], lo, false);
      hi = __builtin_amdgcn_sdot4((int)(((q >> 4) & 0x0F0F0F0Fu) | (((hb >> 4) & 0x03030303u) << 4)), x.xh[i], hi, false);
    }
    lo -= 32 * x.bs_lo;  // sum (q6 - 32) * q8, exact
    hi -= 32 * x.bs_hi;
    const int sh = 8 * ((c & 1) + 2 * a);
    const int sc_lo = (int)(signed char)(p.sc[0] >> sh), sc_hi = (int)(signed char)(p.sc[1] >> sh);
    return h2f(p.d) * x.d8 * ((float)__mul24(sc_lo, lo) + (float)__mul24(sc_hi, hi));  // (|lo|, |hi| <= 16 * 32 * 128)
  }
}

// The rhs planes of a workgroup in LDS: class-major quants (Q4_K rows), quants in element order (Q6_K rows), d | bsums
struct KqLds {
  unsigned *cm, *el;  // nullptr: no rows of that kind
  float* d;
  short* bs;
};
inline __host__ __device__ size_t kq_lds_bytes(int k, bool both) { return (size_t)k * (both ? 2 : 1) + (size_t)(k / 256) * 4 + (size_t)(k / 16) * 2; }
__device__ __forceinline__ KqLds kq_lds(i32x4* lds, int nsb, bool cm, bool el) {
  KqLds l;
  unsigned* q = (unsigned*)lds;
  l.cm = cm ? q : nullptr;
  q += cm ? nsb * 64 : 0;
  l.el = el ? q : nullptr;
  q += el ? nsb * 64 : 0;
  l.d = (float*)q;
  l.bs = (short*)(l.d + nsb);
  return l;
}
__device__ __forceinline__ void kq_quant(const KqLds& l, int sb, const f32x4 v, int lane) {
  const Q8KLane o = q8k_wave_quant(v, lane);
  if (l.cm) q8k_store_class_major((signed char*)(l.cm + sb * 64), lane, o.packed);
  if (l.el) l.el[sb * 64 + lane] = o.packed;
  if ((lane & 3) == 0) l.bs[sb * 16 + (lane >> 2)] = (short)o.quad_sum;
  if (lane == 0) l.d[sb] = o.d;
}
__device__ __forceinline__ ActQ8_K kq_act(const KqLds& l) { return ActQ8_K{(const i32x4*)l.el, l.d, l.bs, (const i32x4*)l.cm}; }

// The rhs is (x / rms) * w: requested ahead of the first weights (loads return in order: behind them it would wait for an HBM round trip instead of an L2
// one), normalized and quantized under them.  Every wave forms the rms for itself from the chunk sums of the launch that left x -- two halves of 16 rows a chunk,
// 64 chunks a round through wave_sum_f32, rounds in order -- which takes a barrier less than sharing it.  U super-blocks a wave at the most, R rounds; requests are
// clamped and never skipped: behind a branch around one the compiler waits for all that are out.
template <int U, int R>
struct KqNorm {
  f32x4 x[U], w[U];
  f32x2 c[R];
};
template <int U, int R>
__device__ __forceinline__ void kq_norm_request(KqNorm<U, R>& n, const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ csums, int nsb, int lane,
                                                int wave, int nw) {
#pragma unroll
  for (int r = 0; r < R; r++) n.c[r] = ((const f32x2*)csums)[r * 64 + lane < nsb * 8 ? r * 64 + lane : nsb * 8 - 1];
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int sb = wave + u * nw < nsb ? wave + u * nw : 0;
    n.x[u] = ((const f32x4*)x)[sb * 64 + lane];
    n.w[u] = ((const f32x4*)w)[sb * 64 + lane];
  }
}
// ORD (strict-order device): rms_norm.rs:35-40's own order -- a chunk's 32 squares as one scan from -0.0, the chunks' sums one after the other.  The first half of every scan comes
// with x (csums); the row goes to LDS (t, in front of the records; chunks 36 floats apart: lanes read their chunks' 16-byte pieces from different banks) and one wave goes on with
// the second halves, a lane a chunk, and adds the sums lane by lane.
inline __host__ __device__ size_t kq_ord_bytes(int nsb) { return (size_t)nsb * 8 * 36 * 4; }
template <int U, int R>
__device__ __forceinline__ float kq_ordered_rms(KqNorm<U, R>& n, float* __restrict__ t, float eps, int nsb, int lane, int wave, int nw) {
  __shared__ __attribute__((aligned(16))) float s_chunk[64 * R];
  __shared__ float s_rms;
  const int nch = nsb * 8;
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int sb = wave + u * nw;
    if (sb < nsb) *(f32x4*)(t + (sb * 8 + (lane >> 3)) * 36 + (lane & 7) * 4) = n.x[u];
  }
  __syncthreads();
  if (wave == 0) {
    float s[R];
#pragma unroll
    for (int r = 0; r < R; r += 2) {  // (two rounds together: their scans hide each other; the first weights are on their way to most registers)
      f32x4 v[2][2];
#pragma unroll
      for (int h = 0; h < 2; h++) s[r + h] = n.c[r + h][0];
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int c = (r + h) * 64 + lane;
#pragma unroll
          for (int i = 0; i < 2; i++) v[h][i] = *(const f32x4*)(t + (c < nch ? c : nch - 1) * 36 + 16 + (j + i) * 4);
        }
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
          for (int h = 0; h < 2; h++) s[r + h] += v[h][i >> 2][i & 3] * v[h][i >> 2][i & 3];
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++) s_chunk[r * 64 + lane] = r * 64 + lane < nch ? s[r] : 0.0f;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    float sum = 0.0f;
    f32x4 q[2];  // (eight sums are read while eight are added; sums past the row are +0.0)
    q[0] = ((const f32x4*)s_chunk)[0];
    q[1] = ((const f32x4*)s_chunk)[1];
#pragma unroll 1
    for (int c = 0; c < nch; c += 8) {
      const float* next = s_chunk + (c + 8 < 64 * R ? c + 8 : 0);
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const f32x4 v = q[i];
        q[i] = ((const f32x4*)next)[i];
        sum += v[0];
        sum += v[1];
        sum += v[2];
        sum += v[3];
      }
    }
    if (lane == 0) s_rms = sqrtf(sum / (float)(nsb * 256) + eps);
  }
  __syncthreads();
  return s_rms;
}
template <int U, int R, bool ORD>
__device__ __forceinline__ void kq_norm_quant(KqNorm<U, R>& n, const KqLds& l, float* __restrict__ t, float eps, int nsb, int lane, int wave, int nw) {
#pragma unroll
  for (int u = 0; u < U; u++) asm volatile("" : "+v"(n.x[u]), "+v"(n.w[u]));  // (else the compiler moves the requests into the branch that uses them)
  float rms;
  if constexpr (ORD) {
    rms = kq_ordered_rms(n, t, eps, nsb, lane, wave, nw);
  } else {
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < R; r++) sum += wave_sum_f32(r * 64 + lane < nsb * 8 ? n.c[r][0] + n.c[r][1] : 0.0f);  // (rounds past the row add +0.0)
    rms = sqrtf(sum / (float)(nsb * 256) + eps);
  }
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int sb = wave + u * nw;
    if (sb >= nsb) break;  // (wave-uniform)
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = (n.x[u][i] / rms) * n.w[u][i];  // rms_norm.rs:41-45, then the weight (llama2.rs:611)
    kq_quant(l, sb, v, lane);
  }
}

// R rows of a wave, P of a lane's pieces of each on their way or there
template <bool SIX, int R, int P>
__device__ __forceinline__ void kq_request(KqPiece<SIX> (&p)[P][R], const KqMat& m, int row0, int last, int nsb, int lane) {
  const int np = nsb * 8;
#pragma unroll
  for (int j = 0; j < P; j++)
#pragma unroll
    for (int r = 0; r < R; r++) p[j][r] = kq_load<SIX>(m, row0 + r < last ? row0 + r : last, nsb, j * 64 + lane < np ? j * 64 + lane : np - 1);
}
template <bool SIX, int R, int P>
__device__ __forceinline__ void kq_rows(KqPiece<SIX> (&p)[P][R], const KqMat& m, const ActQ8_K& act, int row0, int last, int nsb, int lane, float (&acc)[R]) {
  const int np = nsb * 8;
  auto steps = [&](auto More, int c0) {  // More: a piece's registers take the one P further
#pragma unroll
    for (int j = 0; j < P; j++) {
      const int c = c0 + j * 64 + lane, cc = c < np ? c : np - 1;
      if (!decltype(More)::value && c0 + j * 64 >= np) break;  // (uniform)
      const Q4KX x = kq_loadx<SIX>(act, cc);
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float t = kq_term<SIX>(p[j][r], x, cc);
        if (c < np) acc[r] += t;
      }
      if constexpr (decltype(More)::value) {
        const int n = c + P * 64 < np ? c + P * 64 : np - 1;
#pragma unroll
        for (int r = 0; r < R; r++) p[j][r] = kq_load<SIX>(m, row0 + r < last ? row0 + r : last, nsb, n);
      }
    }
  };
  for (int c0 = 0; c0 < np; c0 += P * 64) {
    if (c0 + P * 64 < np)
      steps(std::true_type{}, c0);
    else
      steps(std::false_type{}, c0);
  }
}

// ORD: the rows' records (q4k_class_terms, gemv_core.hpp) to T, `stride` floats a row, a lane a chain adds them (q4k_ordered_sum16)
template <bool SIX>
__device__ __forceinline__ void kq_class_terms(const KqPiece<SIX>& p, const Q4KX& x, int c, bool live, float* __restrict__ t) {
  if constexpr (!SIX) {
    q4k_class_terms<false>(p.w, x, c, live, t);
  } else {
    const int sh = 8 * ((c & 1) + (c & 2));
    q6k_class_terms(p.ql, p.qh, (int)(signed char)(p.sc[0] >> sh), (int)(signed char)(p.sc[1] >> sh), p.d, x.xl, x.xh, x.d8, c, live, t);
  }
}
template <bool SIX, int R, int P>
__device__ __forceinline__ void kq_terms(KqPiece<SIX> (&p)[P][R], const KqMat& m, const ActQ8_K& act, int row0, int last, int nsb, int lane, float* __restrict__ T, int stride) {
  const int np = nsb * 8;
  auto steps = [&](auto More, int c0) {
#pragma unroll
    for (int j = 0; j < P; j++) {
      const int c = c0 + j * 64 + lane, cc = c < np ? c : np - 1;
      if (!decltype(More)::value && c0 + j * 64 >= np) break;  // (uniform)
      const Q4KX x = kq_loadx<SIX>(act, cc);
#pragma unroll
      for (int r = 0; r < R; r++) kq_class_terms<SIX>(p[j][r], x, cc, c < np, T + (size_t)r * stride + (cc >> 3) * 12);
      if constexpr (decltype(More)::value) {
        const int n = c + P * 64 < np ? c + P * 64 : np - 1;
#pragma unroll
        for (int r = 0; r < R; r++) p[j][r] = kq_load<SIX>(m, row0 + r < last ? row0 + r : last, nsb, n);
      }
    }
  };
  for (int c0 = 0; c0 < np; c0 += P * 64) {
    if (c0 + P * 64 < np)
      steps(std::true_type{}, c0);
    else
      steps(std::false_type{}, c0);
  }
}
// floats from the planes on: the records of so many rows, or in front of them the row itself
inline __host__ __device__ size_t kq_rec_at(int k, bool both) { return (kq_lds_bytes(k, both) + 15) & ~(size_t)15; }
inline __host__ __device__ size_t kq_rec_bytes(int rows, int nsb, bool norm) {
  const size_t r = (size_t)rows * q4k_rec_stride(nsb) * 4;
  return norm && kq_ord_bytes(nsb) > r ? kq_ord_bytes(nsb) : r;
}

// Every wave of the workgroup has asked for its share of the rhs before any goes on to weights: a CU takes its waves' requests in turn, 16 cycles each, and the last wave's
// share came 1900 cycles behind the first one's (us a launch without / with: q | k | v 6.2 / 5.8, wo 5.2 / 4.4, ffn_down 9.5 / 9.0; width 2048: wo 3.7 / 3.2, gate | up 6.6 / 6.1).
__device__ __forceinline__ void kq_rhs_first() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

// q | k | v: a wave a pair of rows (the pair that is rotated).  SIX: Q6_K; V6: q and k Q4_K, v Q6_K (*_K_M files).  A workgroup of 4 to 16 waves: one round of workgroups, and a super-block a wave
// where that is up to eight (3072 x 2048 4.5 us with four, 4.0 with eight, 4.4 with twelve; 6144 x 4096 7.7 with eight, 5.8 with twelve, 6.8 with sixteen).
template <bool SIX, bool V6, int U, int R, bool ORD = false>
__global__ __launch_bounds__(1024) void k_kq_qkv(KqMat wq, KqMat wk, KqMat wv, const float* __restrict__ x, const float* __restrict__ wnorm, float eps,
                                                 const float* __restrict__ csums, int nsb, QkvEpi e) {
  extern __shared__ i32x4 lds_act[];
  const int lane = threadIdx.x & 63, wave = wave_in_wg(), nw = blockDim.x >> 6;
  const int v0 = e.dim + e.kv_dim, first = blockIdx.x * nw * 2;
  const KqLds l = kq_lds(lds_act, nsb, !SIX && (!V6 || first < v0), SIX || (V6 && first + nw * 2 > v0));
  const int total = e.dim + 2 * e.kv_dim, want = (blockIdx.x * nw + wave) * 2;
  const bool live = want < total;  // (wave-uniform; a wave without rows stays for its super-blocks)
  const int row0 = live ? want : 0;
  KqMat w = wq;
  int local = row0, m = e.dim;
  bool v6 = false;
  if (row0 >= e.dim) {
    const bool v = row0 >= v0;
    w = v ? wv : wk;
    local = row0 - e.dim - (v ? e.kv_dim : 0);
    m = e.kv_dim;
    v6 = V6 && v;
  }
  KqNorm<U, R> n;
  kq_norm_request(n, x, wnorm, csums, nsb, lane, wave, nw);
  kq_rhs_first();
  const QkvPre pre = qkv_preload_nb(e, row0);
  KqPiece<SIX> p[2][2];
  constexpr int P6 = ORD ? 1 : 2;  // (registers)
  KqPiece<true> p6[V6 ? P6 : 1][V6 ? 2 : 1];
  if (V6 && v6) {
    if constexpr (V6) kq_request<true, 2, P6>(p6, w, local, m - 1, nsb, lane);
  } else {
    kq_request<SIX, 2, 2>(p, w, local, m - 1, nsb, lane);
  }
  float* T = (float*)((char*)lds_act + kq_rec_at(nsb * 256, V6));
  kq_norm_quant<U, R, ORD>(n, l, T, eps, nsb, lane, wave, nw);
  __syncthreads();
  if (!live) return;
  if constexpr (ORD) {
    const int stride = q4k_rec_stride(nsb);
    float* Tw = T + (size_t)wave * 2 * stride;
    if (V6 && v6) {
      if constexpr (V6) kq_terms<true, 2, P6>(p6, w, kq_act(l), local, m - 1, nsb, lane, Tw, stride);
    } else {
      kq_terms<SIX, 2, 2>(p, w, kq_act(l), local, m - 1, nsb, lane, Tw, stride);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    const float s = q4k_ordered_sum16(Tw + (size_t)(lane >> 4 & 1) * stride, nsb, lane);
    const float s1 = rl_f(s, 16);
    if (lane == 0) qkv_epilogue(e, pre, row0, s, s1);
    return;
  }
  float acc[2] = {0.f, 0.f};
  if (V6 && v6) {
    if constexpr (V6) kq_rows<true, 2, P6>(p6, w, kq_act(l), local, m - 1, nsb, lane, acc);
  } else {
    kq_rows<SIX, 2, 2>(p, w, kq_act(l), local, m - 1, nsb, lane, acc);
  }
  const float s0 = wave_sum_f32(acc[0]), s1 = wave_sum_f32(acc[1]);
  if (lane == 0) qkv_epilogue(e, pre, row0, s0, s1);
}

// gate | up + SiLU * mul: two rows of each a wave, 32 a workgroup of sixteen waves, two of them a CU (64 registers; one where the records of long rows fill its LDS); h leaves as f32
template <bool SIX, int U, int R, bool ORD = false>
__global__ __launch_bounds__(1024, ORD && U > 1 ? 4 : 8) void k_kq_gateup(KqMat wg, KqMat wu, const float* __restrict__ x, const float* __restrict__ wnorm, float eps,
                                                       const float* __restrict__ csums, int nsb, const unsigned short* __restrict__ exp_tab, float* __restrict__ h, int m) {
  extern __shared__ i32x4 lds_act[];
  const KqLds l = kq_lds(lds_act, nsb, !SIX, SIX);
  const int lane = threadIdx.x & 63, wave = wave_in_wg();
  const int row0 = (blockIdx.x * 16 + wave) * 2;
  KqNorm<U, R> n;
  kq_norm_request(n, x, wnorm, csums, nsb, lane, wave, 16);
  kq_rhs_first();
  KqPiece<SIX> p[1][2];
  kq_request<SIX, 2, 1>(p, wg, row0, m - 1, nsb, lane);
  float* T = (float*)((char*)lds_act + kq_rec_at(nsb * 256, false));  // rows 0 .. 31: gate, 32 .. 63: up
  kq_norm_quant<U, R, ORD>(n, l, T, eps, nsb, lane, wave, 16);
  __syncthreads();
  const ActQ8_K act = kq_act(l);
  if constexpr (ORD) {  // (host: m is a multiple of 32)
    const int stride = q4k_rec_stride(nsb);
    kq_terms<SIX, 2, 1>(p, wg, act, row0, m - 1, nsb, lane, T + (size_t)wave * 2 * stride, stride);
    kq_request<SIX, 2, 1>(p, wu, row0, m - 1, nsb, lane);
    kq_terms<SIX, 2, 1>(p, wu, act, row0, m - 1, nsb, lane, T + (size_t)(32 + wave * 2) * stride, stride);
    __syncthreads();
    if (wave != 0) return;
    const float s = q4k_ordered_sum<3>(T + (size_t)lane * stride, nsb);  // (three records ahead: a fourth does not fit the 64 registers.  A lane a chain: 19.3 us, not 19.0)
    const float u = __shfl(s, (lane & 31) + 32, 64);
    if (lane < 32) h[(int)blockIdx.x * 32 + lane] = silu_mul(s, u, exp_tab);
    return;
  }
  if (row0 >= m) return;
  float ag[2] = {0.f, 0.f}, au[2] = {0.f, 0.f};
  kq_rows<SIX, 2, 1>(p, wg, act, row0, m - 1, nsb, lane, ag);
  kq_request<SIX, 2, 1>(p, wu, row0, m - 1, nsb, lane);
  kq_rows<SIX, 2, 1>(p, wu, act, row0, m - 1, nsb, lane, au);
#pragma unroll
  for (int r = 0; r < 2; r++) {
    const float g = wave_sum_f32(ag[r]), u = wave_sum_f32(au[r]);
    if (lane == 0 && row0 + r < m) h[row0 + r] = silu_mul(g, u, exp_tab);
  }
}

// the end of a workgroup's 16 rows: hv their dots, res what they are added to; one wave
__device__ __forceinline__ void kq_res_out(float* hv, float res, float* __restrict__ x, float* __restrict__ csums, int lane) {
  if (lane < 16) {
    const float xv = hv[lane] + res;  // x = matmul_out + x (llama2.rs:266 / :636)
    x[blockIdx.x * 16 + lane] = xv;
    hv[lane] = xv;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  float cs = -0.0f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const f32x4 t = ((const f32x4*)hv)[j];
    cs += t[0] * t[0];
    cs += t[1] * t[1];
    cs += t[2] * t[2];
    cs += t[3] * t[3];
  }
  if (lane == 0) csums[blockIdx.x] = cs;
}
// wo, ffn_down: x += W . quantized(in), a row a wave, 16 a workgroup; the workgroup's sum of squares of x goes to csums (a plain store, read by the next launch)
template <bool SIX, int U, int P, bool ORD = false>
__global__ __launch_bounds__(1024) void k_kq_res(KqMat w, const float* __restrict__ in, int nsb, float* __restrict__ x, float* __restrict__ csums) {
  extern __shared__ i32x4 lds_act[];
  __shared__ __attribute__((aligned(16))) float hv[16];
  const KqLds l = kq_lds(lds_act, nsb, !SIX, SIX);
  const int lane = threadIdx.x & 63, wave = wave_in_wg(), row = blockIdx.x * 16 + wave;
  f32x4 v[U];
#pragma unroll
  for (int u = 0; u < U; u++) v[u] = ((const f32x4*)in)[(wave + u * 16 < nsb ? wave + u * 16 : 0) * 64 + lane];
  KqPiece<SIX> p[P][1];
  kq_rhs_first();
  kq_request<SIX, 1, P>(p, w, row, row, nsb, lane);
  const float res = x[blockIdx.x * 16 + (lane & 15)];  // (wave 0's; no branch)
#pragma unroll
  for (int u = 0; u < U; u++) asm volatile("" : "+v"(v[u]));  // (as in kq_norm_quant)
#pragma unroll
  for (int u = 0; u < U; u++) {
    if (wave + u * 16 >= nsb) break;  // (wave-uniform)
    kq_quant(l, wave + u * 16, v[u], lane);
  }
  for (int sb = wave + U * 16; sb < nsb; sb += 16) kq_quant(l, sb, ((const f32x4*)in)[sb * 64 + lane], lane);
  __syncthreads();
  if constexpr (ORD) {
    const int stride = q4k_rec_stride(nsb);
    float* T = (float*)((char*)lds_act + kq_rec_at(nsb * 256, false));
    kq_terms<SIX, 1, P>(p, w, kq_act(l), row, row, nsb, lane, T + (size_t)wave * stride, stride);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    const float s = q4k_ordered_sum16(T + (size_t)wave * stride, nsb, lane);
    if (lane == 0) hv[wave] = s;
    __syncthreads();
    if (wave != 0) return;
    kq_res_out(hv, res, x, csums, lane);
    return;
  }
  float acc[1] = {0.f};
  kq_rows<SIX, 1, P>(p, w, kq_act(l), row, row, nsb, lane, acc);
  const float s = wave_sum_f32(acc[0]);
  if (lane == 0) hv[wave] = s;
  __syncthreads();
  if (wave != 0) return;
  kq_res_out(hv, res, x, csums, lane);
}

}  // namespace crabml_hip
