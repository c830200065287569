// gemm_f16.hip -- f16 rows x f16 weights on the matrix cores: the linears of a prompt pass and matmul_vec's batched rhs of many results where
// the weights are F16 (fast device; buf_f16.rs:83-97: the rhs is rounded to f16, products are exact in f32, sums are f32).
//
//   out[m][row][n] = sum_k a[row][k] w[m][n][k]     up to three matrices of one rhs (q | k | v, gate | up) in one launch
//
// Bound: v_mfma_f32_16x16x32_f16 issue and the LDS reads that feed it.  The tiles, the loads straight into LDS and the cut of k are those
// of gemm_bf16.hip; what differs is that the operands are the caller's own buffers without padding: a row past the end is the last one
// again (its results are not stored), a 16-byte piece past the end of k is a piece of zeros.  Weights are the first operand, so that a
// lane's four results are neighbouring columns of one row and leave as one 16-byte store, without a way through LDS.
//
// Measured (203 rows, width 2048, ff 8192, one layer): q | k | v 15.4 us, wo 15.0, gate | up 28.1, ff_down 29.4 (490 TFLOP/s in the
// gate | up launch); 17.8, 17.2, 33.6, 28.5 with a step's requests in a row behind its barrier and four waves on a 128-row tile (ff_down, on 64-row
// tiles in pieces of k, gained nothing).
#include <type_traits>

#include "gemm_bf16.hpp"

namespace crabml_hip {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __attribute__((aligned(16))) unsigned short g_zero_piece[8];  // (never written)

template <int BM, int BN, int WGM, int WGN, int ST>
__global__ __launch_bounds__(64 * WGM * WGN) void k_gemm_f16(const GemmF16 g, int S, float* __restrict__ ws, unsigned* __restrict__ tick) {
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
  constexpr int NT = 64 * WGM * WGN, FA = BM * 8 / NT, FB = BN * 8 / NT;  // threads; a step's requests per thread
  static_assert(WM % 16 == 0 && WN % 16 == 0 && BM * 8 % NT == 0 && BN * 8 % NT == 0, "whole fragments, whole requests");
  __shared__ __attribute__((aligned(16))) unsigned short lds[ST][(BM + BN) * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg();
  const int wm = wave / WGN, wn = wave % WGN;
  const int mt = (g.M + BM - 1) / BM, nt = g.end[2], total = mt * nt * S;
  int id = blockIdx.x;
  {  // XCD x (= id % 8) takes a contiguous run of tiles
    const int x = id & 7, i = id >> 3, q = total >> 3, r = total & 7;
    id = x * q + (x < r ? x : r) + i;
  }
  const int piece = id / mt % S, tile = id / mt / S * mt + id % mt;
  const int row0 = (tile % mt) * BM, ct = tile / mt;
  const int mat = ct < g.end[0] ? 0 : ct < g.end[1] ? 1 : 2;
  const int col0 = (ct - (mat == 0 ? 0 : g.end[mat - 1])) * BN, N = g.n[mat];
  const unsigned short* pa[FA];
  const unsigned short* pb[FB];
  const int c8 = ((tid & 7) ^ ((tid >> 4) & 7)) * 8;  // this thread's piece of a step's 64 (the permutation has a period of 16 rows)
  static_assert(NT / 8 % 16 == 0, "every request of a thread takes the same piece");
#pragma unroll
  for (int it = 0; it < FA; it++) {
    const int r = row0 + (it * NT + tid) / 8;
    pa[it] = (const unsigned short*)((const char*)g.a + (size_t)(r < g.M ? r : g.M - 1) * g.a_stride) + c8;
  }
#pragma unroll
  for (int it = 0; it < FB; it++) {
    const int r = col0 + (it * NT + tid) / 8;
    pb[it] = g.w[mat] + (size_t)(r < N ? r : N - 1) * g.K + c8;
  }
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (g.K + 63) / 64;
  const int s_lo = (int)((long long)steps * piece / S), s_hi = (int)((long long)steps * (piece + 1) / S);
  constexpr unsigned STAGE = (BM + BN) * 128;  // bytes of a step
  const unsigned lds0 = lds_address(&lds[0][wave * 512]);
  auto request = [&](int s, unsigned into, int i) {  // step s's request i of FA + FB
    const int k0 = s * 64;
    const bool in = k0 + c8 < g.K;  // (K is a multiple of 8)
    lds_dma16(in ? (i < FA ? pa[i < FA ? i : 0] : pb[i < FA ? 0 : i - FA]) + k0 : g_zero_piece, into + i * NT * 16);
  };
  const int fr = lane & 15, fk = lane >> 4;
#pragma unroll
  for (int i = 0; i < ST - 1; i++)
    if (s_lo + i < s_hi) {
#pragma unroll
      for (int d = 0; d < FA + FB; d++) request(s_lo + i, lds0 + i * STAGE, d);
    }
  int buf = 0;  // the stage that step s is in
  auto step = [&](auto Mc, int s) {
    const unsigned into = lds0 + (buf == 0 ? ST - 1 : buf - 1) * STAGE;
    tile_step<f16x8, TM, TN, decltype(Mc)::value ? FA + FB : 0>(
        &lds[buf][0], wm * WM, &lds[buf][BM * 64], wn * WN,
        [&](int i, int j, f16x8 x, f16x8 y) { acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(y, x, acc[i][j], 0, 0, 0); },
        [&](int d) { request(s + ST - 1, into, d); });
    buf = buf + 1 == ST ? 0 : buf + 1;
  };
  int s = s_lo;
  for (; s + ST - 1 < s_hi; s++) {
    landed_barrier<(ST - 2) * (FA + FB)>();
    step(std::true_type{}, s);
  }
  for (; s < s_hi; s++) {
    if (s + ST - 2 < s_hi)
      landed_barrier<(ST - 2) * (FA + FB)>();
    else
      landed_barrier<0>();
    step(std::false_type{}, s);
  }
  if (S > 1 && !add_pieces<TM * TN, NT>((f32x4*)acc, S, piece, tile, ws, tick)) return;
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int row = row0 + wm * WM + i * 16 + fr;
    if (row >= g.M) continue;
    float* o = g.out[mat] + (size_t)row * N;
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int col = col0 + wn * WN + j * 16 + fk * 4;
      if (N % 4 == 0) {
        if (col < N) *(f32x4*)(o + col) = acc[i][j];
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (col + e < N) o[col + e] = acc[i][j][e];
      }
    }
  }
}

bool launch_gemm_f16(crabml_hip_device* dev, crabml_hip_device::ProfRec* rec, const void* const* w, const size_t* n, int nw, size_t k,
                     const void* act, size_t act_stride, size_t rows, float* const* out, const GemmScratch& ws) {
  if (nw < 1 || nw > 3 || rows < 2 || k == 0 || k % 8 != 0 || act_stride % 16 != 0 || (size_t)act % 16 != 0) return false;
  if (rows > (1u << 20) || k > (1u << 24)) return false;
  GemmF16 g;
  g.a = act;
  g.a_stride = act_stride;
  g.M = (int)rows;
  g.K = (int)k;
  int tiles = 0;
  for (int i = 0; i < 3; i++) {
    if (i < nw) {
      if (n[i] == 0 || n[i] > (1u << 24) || (size_t)w[i] % 16 != 0 || (size_t)out[i] % 16 != 0) return false;
      g.w[i] = (const unsigned short*)w[i];
      g.out[i] = out[i];
      g.n[i] = (int)n[i];
      tiles += (int)((n[i] + 127) / 128);
    }
    g.end[i] = tiles;
  }
  const GemmPlan p = gemm_plan(g.M, tiles, (g.K + 63) / 64, dev->n_cu, ws.partials ? ws.floats : 0);
  const dim3 grid((unsigned)(((g.M + p.bm - 1) / p.bm) * tiles * p.S));
  hipStream_t st = dev->stream;
  if (p.bm == 256)
    launch_k(st, rec, k_gemm_f16<256, 128, 4, 2, 3>, grid, dim3(512), 0, g, p.S, ws.partials, ws.ticks);
  else if (p.bm == 128)
    launch_k(st, rec, k_gemm_f16<128, 128, 4, 2, 4>, grid, dim3(512), 0, g, p.S, ws.partials, ws.ticks);
  else if (p.bm == 64)
    launch_k(st, rec, k_gemm_f16<64, 128, 2, 2, 3>, grid, dim3(256), 0, g, p.S, ws.partials, ws.ticks);
  else
    launch_k(st, rec, k_gemm_f16<32, 128, 2, 2, 4>, grid, dim3(256), 0, g, p.S, ws.partials, ws.ticks);
  return true;
}

}  // namespace crabml_hip
