// gemm_f16w_wide.hip -- the fast prompt pass's weight GEMM (gemm_f16w.hip: operands, formats, k-slot orders) for passes of more than 64 rows whose k
// is a multiple of 256, where the launch has workgroups enough (f16w_takes_wide).
//
// What bounds it: the matrix cores, if everything beside them stays out of their way.  gemm_f16w.hip's waves hold two 16-row fragments, so every B'
// fragment read from LDS feeds two products: 8 waves read 64 KB per 32 slots of k, the 512 cycles that their products take.  Here
//  - a wave of the wide tile holds F = 4 fragments x T column tiles (128 accumulators a lane, still two waves a SIMD): half the reads a product;
//  - B' goes from memory straight into LDS (no registers, no LDS writes by the waves), two chunks deep;
//  - A's quants are asked for a chunk ahead WITHOUT a streaming hint: the column tiles of a row tile run side by side on an XCD, and with the
//    hint each of them fetched its own copy (gate | up of 512 rows, 14336 x 4096 Q4_0, F = 4: 176 us with, 146 without);
//  - the scales of two chunks -- 16 bytes of a row in every format -- come by one request of 64 rows into LDS: as two-byte gathers they took a
//    line per row and chunk from L2, as much traffic as the quants (146 -> 124 us);
//  - few tiles: KG = 2 groups of waves in a workgroup take half of k each and add their accumulators through LDS, where pieces of k in memory cost
//    a write and a read of the output each (4096 x 4096, 512 rows: 40.6 -> 30.1 us with both).
// Measured against gemm_f16w.hip, Q4_0 (Q8_0), us: gate | up of 512 rows 165 -> 124 (194 -> 141), 1024 rows 330 -> 239 (388 -> 261); q | k | v of 512 rows
// 55.7 -> 38.0, wo 40.5 -> 30.1, ffn_down 110 -> 72; ffn_down of 1024 rows 173 -> 131.  What is left of gate | up beside its products (58 us at the clock
// that the chip holds): the unpacking (17), the requests (15), SiLU's table (8).
#include <type_traits>

#include "gemm_f16w.hpp"
#include "lds_dma.hpp"

namespace crabml_hip {

// LDS: two buffers of [k group][column][256 bytes]: a column's sixteen 16-byte pieces (block g of the chunk, step s: 4 g + s), piece p at
// p ^ wide_swizzle(column), so that the 16 lanes which ds_read_b128 serves together (columns 0-3 and 12-15 of one g with 4-11 of the next) touch
// all 64 banks once.  Then each wave's scales: two slots of [row][16 bytes].
__device__ __forceinline__ int wide_swizzle(int c) { return (c & 3) | ((c & 8) ? 12 : 0); }

template <int F, int T, int KG>
struct WideGeo {
  static constexpr int RW = 4, CW = 16 * T, NT = 64 * RW * KG;  // waves along the rows, columns, threads
  static constexpr int BUF = CW * 256, SCALES = 2 * KG * BUF;   // bytes of a chunk of B' of one k group; where the scales begin
  static constexpr int DMA = CW * 16 / (64 * RW);               // requests of B' a thread and chunk
  static constexpr int STAGE = SCALES + RW * KG * 2048;
  static constexpr int SUMS = (KG - 1) * RW * T * F * 1024;     // accumulators on their way to another k group
  static constexpr int H_ROWS = 16 * RW * (F / 2), H_STRIDE = H_ROWS + 4;  // gate | up: h of the workgroup (four banks between columns)
  static constexpr int ENDS = SUMS + CW * H_STRIDE * 4;
  static constexpr int LDS_BYTES = STAGE > ENDS ? STAGE : ENDS;
};

// F 16-row fragments x T 16-column tiles per wave; four waves along the rows, KG groups of them along k.  GU: fragments 0 .. F/2 - 1 are rows of
// the first matrix, the others the same rows of the second, and the epilogue stores h = silu(g) * u (gemm_f16w.hip).
template <int WF, int F, int T, int KG, bool GU>
__global__ __launch_bounds__(256 * KG, 2) void k_gemm_f16w_wide(F16wMats mats, const char* __restrict__ xh, int nb, int n, int row_tiles, int ksplit) {
  using G = WideGeo<F, T, KG>;
  constexpr int RW = G::RW, CW = G::CW, BUF = G::BUF, DMA = G::DMA;
  constexpr int FR = GU ? F / 2 : F;                               // fragments of consecutive rows
  constexpr int NQ = (WF == WF_Q8_0 || WF == WF_Q6_K) ? 2 : 1;     // 16-byte quant loads per fragment and chunk
  extern __shared__ __attribute__((aligned(16))) unsigned char wide_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg();
  const int rw = wave % RW, kg = wave / RW;
  const int i = lane & 15, g = lane >> 4;
  int rt, ct, ks;
  {  // XCD x (= id % 8) takes a contiguous run of (row tile, piece of k, column tile): a row tile's readers are neighbours on one L2
    const int total = (int)gridDim.x, per_row = total / row_tiles, col_tiles = per_row / ksplit;
    const int x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3, q = total >> 3, r = total & 7;
    const int id = x * q + (x < r ? x : r) + j;
    rt = id / per_row;
    const int sub = id - rt * per_row;
    ks = sub / col_tiles;
    ct = sub - ks * col_tiles;
  }
  const int ti = GU ? 0 : rt < mats.tiles_end[0] ? 0 : rt < mats.tiles_end[1] ? 1 : 2;  // (uniform)
  const int m = ti == 0 ? mats.m[0] : ti == 1 ? mats.m[1] : mats.m[2];
  const int rt_l = rt - (ti == 0 ? 0 : ti == 1 ? mats.tiles_end[0] : mats.tiles_end[1]);
  const int r0 = (rt_l * RW + rw) * 16 * FR, c0 = ct * CW;
  // this k group's chunks of 128 slots: [ch_lo, ch_lo + nchunks), whole pairs (nchunks <= 0: none, behind the last piece's end)
  const int all_chunks = nb >> 2, pieces = KG * ksplit;
  const int per_piece = ((all_chunks + pieces - 1) / pieces + 1) & ~1;
  const int ch_lo = (ks * KG + kg) * per_piece;
  const int nchunks = all_chunks - ch_lo < per_piece ? all_chunks - ch_lo : per_piece;

  // A: chunk c + 1 is asked for while chunk c is multiplied (the two register sets are compile-time: the chunk loop is unrolled by two)
  const char* wq[GU ? 2 : 1];  // (uniform)
  const char* wh[GU ? 2 : 1];  // Q6_K: the high bits
  const unsigned short* wd[GU ? 2 : 1];
#pragma unroll
  for (int u = 0; u < (GU ? 2 : 1); u++) {
    const int j = GU ? u : ti;
    wq[u] = (const char*)(j == 0 ? mats.wq[0] : j == 1 ? mats.wq[1] : mats.wq[2]);
    wh[u] = j == 0 ? mats.wd[0] : j == 1 ? mats.wd[1] : mats.wd[2];
    wd[u] = (const unsigned short*)(j == 0 ? mats.ws3[0] : j == 1 ? mats.ws3[1] : mats.ws3[2]);
  }
  unsigned row_of[F];  // (below 2^32 bytes of quants: the launcher's check)
#pragma unroll
  for (int f = 0; f < F; f++) {
    const int row = r0 + 16 * (f % FR) + i;
    row_of[f] = (unsigned)(row < m ? row : m - 1);
  }
  i32x4 aq[2][NQ * F];
  unsigned hd[F];  // Q6_K: d of the pair's super-block
  auto fetch_a = [&](auto Jc, int ch, int f) {  // (past the end: the last chunk again, never consumed)
    constexpr int J = decltype(Jc)::value;
    const unsigned cc = (unsigned)(ch_lo + (ch < nchunks ? ch : nchunks - 1));
    const int u = GU && f >= FR ? 1 : 0;
    if constexpr (WF == WF_Q4_K) {
      aq[J][f] = *(const i32x4*)(wq[u] + (row_of[f] * (unsigned)(nb * 16) + (cc >> 1) * 128u + (unsigned)(J * 16 + 32 * g)));
    } else if constexpr (WF == WF_Q6_K) {
      aq[J][2 * f] = *(const i32x4*)(wq[u] + (row_of[f] * (unsigned)(nb * 16) + cc * 64u + (unsigned)(16 * g)));
      aq[J][2 * f + 1] = *(const i32x4*)(wh[u] + (row_of[f] * (unsigned)(nb * 8) + cc * 32u + (unsigned)(16 * (g & 1))));
      if constexpr (J == 0) hd[f] = wd[u][row_of[f] * (unsigned)(nb >> 3) + (cc >> 1)];
    } else {
#pragma unroll
      for (int q = 0; q < NQ; q++)
        aq[J][NQ * f + q] = *(const i32x4*)(wq[u] + (row_of[f] * (unsigned)(nb * 16 * NQ) + cc * (64u * NQ) + (unsigned)(16 * NQ * g + 16 * q)));
    }
  };
  // scales: lane l asks for the 16 bytes of row l of the wave's 16 F (F = 2: the upper lanes repeat the lower ones)
  constexpr int SROW = WF == WF_Q4_1 ? 4 : 2;  // bytes a block
  unsigned char* const sc = wide_lds + G::SCALES + wave * 2048;
  const unsigned sc_at = lds_address(sc);
  const char* srow;
  {
    const int f = (lane >> 4) % F, u = GU && f >= FR ? 1 : 0, row = r0 + 16 * (f % FR) + i;
    const char* p0 = WF == WF_Q6_K ? (ti == 0 ? mats.ws2[0] : ti == 1 ? mats.ws2[1] : mats.ws2[2]) : wh[0];
    const char* p1 = !GU ? p0 : WF == WF_Q6_K ? mats.ws2[1] : wh[GU ? 1 : 0];
    srow = (u ? p1 : p0) + (size_t)(row < m ? row : m - 1) * nb * SROW;
  }
  auto fetch_s = [&](int ch) {  // a pair of chunks from an even one on (Q4_1: one chunk)
    if constexpr (WF == WF_Q4_1)
      lds_dma16(srow + (size_t)(ch_lo + (ch < nchunks ? ch : nchunks - 1)) * 16, sc_at + (ch & 1) * 1024);
    else
      lds_dma16(srow + (size_t)(ch_lo + (ch < nchunks ? ch : nchunks - 2)) * 8, sc_at + ((ch >> 1) & 1) * 1024);
  };
  // B': request d asks for 16 columns; a thread's column and piece of it.  Columns past n read what follows in xh (inside its allocation: gemm_f16w_xh_bytes)
  const int tg = tid - kg * (64 * RW);
  const unsigned xoff = (unsigned)(tg >> 4) * (unsigned)nb * 64u + (unsigned)(((tg & 15) ^ wide_swizzle(tg >> 4)) * 16);
  const char* xbase = xh + (size_t)c0 * nb * 64 + (size_t)ch_lo * 256;  // (uniform in a wave, as ch_lo)
  const unsigned b_at = lds_address(wide_lds + kg * BUF + rw * 1024);
  auto fetch_b = [&](int buf, int ch, int d) {
    lds_dma16(xbase + (ptrdiff_t)(ch < nchunks ? ch : nchunks - 1) * 256 + (size_t)d * nb * 1024, xoff, b_at + buf * (KG * BUF) + d * (RW * 1024));
  };

  f32x4 acc[F][T];
#pragma unroll
  for (int f = 0; f < F; f++)
#pragma unroll
    for (int t = 0; t < T; t++) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned magic = 0x64006400u;
  asm volatile("" : "+v"(magic));  // pinned in a VGPR (and_or_magic)
#pragma unroll
  for (int d = 0; d < DMA; d++) fetch_b(0, 0, d);
#pragma unroll
  for (int f = 0; f < F; f++) fetch_a(std::integral_constant<int, 0>{}, 0, f);
  fetch_s(0);
  int piece_at[4];  // of the lane's column and block, by step
#pragma unroll
  for (int s = 0; s < 4; s++) piece_at[s] = i * 256 + (((4 * g + s) ^ wide_swizzle(i)) * 16);
  f16x2 d2[F];         // Q4_0, Q8_0
  Q4KF16Consts cs[F];  // Q4_K: of the pair's super-block; Q4_1: (d, m); Q6_K: d sc of the chunk's half

  // B' fragments in groups of TG tiles: group q + 1 is read while group q is multiplied; the scheduling barriers keep it that way
  constexpr int TG = 2, GS = T / TG, NG = 4 * GS;
  static_assert(T % TG == 0, "whole groups");
  auto products = [&](auto Jc, int ch) {
    constexpr int J = decltype(Jc)::value;
    const unsigned char* S = wide_lds + (J * KG + kg) * BUF;
    f16x8 a[F], bq[2][TG];
    // (used here, behind the barrier's wait: the compiler counts its own requests only, and a wait of its own further down would take in the next chunk's)
#pragma unroll
    for (int u = 0; u < NQ * F; u++) asm volatile("" : "+v"(aq[J][u]));
    if constexpr (WF == WF_Q6_K && J == 0) {
#pragma unroll
      for (int f = 0; f < F; f++) asm volatile("" : "+v"(hd[f]));
    }
    auto read_group = [&](f16x8 (&dst)[TG], int q) {
      const int s = q / GS, t0 = (q % GS) * TG;
#pragma unroll
      for (int t = 0; t < TG; t++) dst[t] = *(const f16x8*)(S + (t0 + t) * 16 * 256 + piece_at[s]);
    };
    read_group(bq[0], 0);
    const unsigned char* sl = sc + (WF == WF_Q4_1 ? J : (ch >> 1) & 1) * 1024 + i * 16;
#pragma unroll
    for (int f = 0; f < F; f++) {
      const unsigned char* p = sl + f * 256;
      if constexpr (WF == WF_Q4_K) {
        if constexpr (J == 0) cs[f] = q4k_f16_consts(*(const i32x4*)p, g);
      } else if constexpr (WF == WF_Q6_K) {
        // the lane's two scales of a half: sc[8 half + (g & 1) + 2 (g >> 1)] (low nibbles' quarter) and 4 further (high nibbles')
        const float d = h2f((unsigned short)hd[f]);
        const signed char* q = (const signed char*)p + 8 * J + (g & 1) + 2 * (g >> 1);
        const _Float16 lo = (_Float16)(d * (float)q[0]), hi = (_Float16)(d * (float)q[4]);
        cs[f].c_lo = f16x2{lo, lo};
        cs[f].c_hi = f16x2{hi, hi};
      } else if constexpr (WF == WF_Q4_1) {
        const unsigned dm = *(const unsigned*)(p + g * 4);
        cs[f].c_lo = cs[f].c_hi = __builtin_bit_cast(f16x2, (dm & 0xffffu) | (dm << 16));
        cs[f].o_lo = cs[f].o_hi = __builtin_bit_cast(f16x2, (dm >> 16) | (dm & 0xffff0000u));
      } else {
        const unsigned d = *(const unsigned short*)(p + J * 8 + g * 2);
        d2[f] = __builtin_bit_cast(f16x2, d | (d << 16));
      }
    }
#pragma unroll
    for (int q = 0; q < NG; q++) {
      const int s = q / GS, t0 = (q % GS) * TG;
      if (q + 1 < NG) read_group(bq[(q + 1) & 1], q + 1);
      constexpr int NR = F + DMA, EV = NG / 2;  // the next chunk's requests, spread over the first half of the products
      if (q < EV) {
#pragma unroll
        for (int r = NR * q / EV; r < NR * (q + 1) / EV; r++) {
          if (r < F)
            fetch_a(std::integral_constant<int, 1 - J>{}, ch + 1, r);
          else
            fetch_b(1 - J, ch + 1, r - F);
        }
      }
      if (q == 0 && (J == 1 || WF == WF_Q4_1)) fetch_s(ch + 1);
      if (q % GS == 0) {
#pragma unroll
        for (int f = 0; f < F; f++) {
          if constexpr (WF == WF_Q4_0) a[f] = unpack_q4_0_f16((unsigned)aq[J][f][s], d2[f], magic);
          if constexpr (WF == WF_Q8_0) a[f] = unpack_q8_0_f16((unsigned)aq[J][2 * f][s], (unsigned)aq[J][2 * f + 1][s], d2[f], magic);
          if constexpr (WF == WF_Q4_K || WF == WF_Q4_1) a[f] = unpack_q4_k_f16((unsigned)aq[J][f][s], cs[f], magic);
          if constexpr (WF == WF_Q6_K)
            a[f] = unpack_q6_k_f16((unsigned)aq[J][2 * f][s], (unsigned)aq[J][2 * f + 1][s] >> (2 * (g >> 1)), cs[f].c_lo, cs[f].c_hi, magic);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < TG; t++)
#pragma unroll
        for (int f = 0; f < F; f++) acc[f][t0 + t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[f], bq[q & 1][t], acc[f][t0 + t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto chunk = [&](auto Jc, int ch) {
    landed_barrier<0>();  // what this chunk reads has landed -- all of it was asked for a chunk of products ago -- and the other buffer has been read by all
    if (KG == 1 || ch < nchunks) products(Jc, ch);
  };
  const int loop = KG == 1 ? nchunks : per_piece;  // (every wave of the workgroup takes the same barriers)
  for (int ch = 0; ch < loop; ch += 2) {
    chunk(std::integral_constant<int, 0>{}, ch);
    chunk(std::integral_constant<int, 1>{}, ch + 1);
  }
  landed_barrier<0>();  // (the requests past the end; LDS is free)

  // D: lane (i, g) holds rows 4 g .. 4 g + 3 of column i of every tile
  float* __restrict__ out = ks == 0 ? (ti == 0 ? mats.out[0] : ti == 1 ? mats.out[1] : mats.out[2])
                                    : (ti == 0 ? mats.out2[0] : ti == 1 ? mats.out2[1] : mats.out2[2]) + (size_t)(ks - 1) * mats.pstride;
  auto store = [&](int f, int t, f32x4 v) {
    const int col = c0 + 16 * t + i, row = r0 + 16 * f + 4 * g;
    if (col < n && row < m) *(f32x4*)(out + (size_t)col * m + row) = v;  // (m % 4 == 0)
  };
  float* const H = (float*)(wide_lds + G::SUMS);
  const bool quant = GU && mats.hq.planes != nullptr;  // (uniform)
  auto finish = [&](int t, const f32x4 (&v)[F]) {
    if constexpr (GU) {
#pragma unroll
      for (int f = 0; f < FR; f++) {
        f32x4 hv;
#pragma unroll
        for (int r = 0; r < 4; r++) hv[r] = f16w_silu_mul(v[f][r], v[f + FR][r], mats.exp_tab);
        if (quant)
          *(f32x4*)(H + (16 * t + i) * G::H_STRIDE + (rw * FR + f) * 16 + 4 * g) = hv;
        else
          store(f, t, hv);
      }
    } else {
#pragma unroll
      for (int f = 0; f < F; f++) store(f, t, v[f]);
    }
  };
  if constexpr (KG == 1) {
#pragma unroll
    for (int t = 0; t < T; t++) {
      f32x4 v[F];
#pragma unroll
      for (int f = 0; f < F; f++) v[f] = acc[f][t];
      finish(t, v);
    }
  } else {
    // each of the two k groups finishes half of the tiles: the other's accumulators of those come through LDS
    constexpr int TK = T / 2;
    static_assert(KG == 2 && T % 2 == 0, "halves");
    f32x4* R = (f32x4*)wide_lds + (size_t)rw * (T * F * 64) + lane;  // [tile][fragment][lane]
#pragma unroll
    for (int t = 0; t < T; t++)
      if (t / TK != kg) {
#pragma unroll
        for (int f = 0; f < F; f++) R[(t * F + f) * 64] = acc[f][t];
      }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T; t++)
      if (t / TK == kg) {
        f32x4 v[F];
#pragma unroll
        for (int f = 0; f < F; f++) v[f] = acc[f][t] + R[(t * F + f) * 64];
        finish(t, v);
      }
  }
  if constexpr (GU) {
    if (quant) {
      __syncthreads();
      f16w_quantize_h<G::H_ROWS / 32, CW, G::H_STRIDE, G::NT>(H, mats.hq, c0, n, rt_l * (G::H_ROWS / 32), m);
    }
  }
}

// hipFuncAttributeMaxDynamicSharedMemorySize, once per (device, kernel)
static bool wide_raise_lds(const crabml_hip_device* dev, const void* fn, int bytes) {
  static std::mutex mu;
  static std::map<std::pair<int, const void*>, bool> have;
  std::lock_guard<std::mutex> g(mu);
  bool& done = have[{dev->ordinal, fn}];
  if (!done && hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
  return done = true;
}
template <int WF, int F, int T, int KG, bool GU>
static bool launch_wide_t(crabml_hip_device* dev, F16wMats& mats, const size_t* m, int nw, size_t k, const void* xh, size_t b, int ksplit) {
  using G = WideGeo<F, T, KG>;
  if (!wide_raise_lds(dev, (const void*)k_gemm_f16w_wide<WF, F, T, KG, GU>, G::LDS_BYTES)) {
    (void)hipGetLastError();
    return false;
  }
  const size_t rows = 16 * G::RW * (GU ? F / 2 : F);
  int row_tiles = 0;
  for (int j = 0; j < 3; j++) {
    if (j < (GU ? 1 : nw)) row_tiles += (int)((m[j] + rows - 1) / rows);
    mats.tiles_end[j] = row_tiles;
  }
  const int col_tiles = (int)((b + G::CW - 1) / G::CW);
  k_gemm_f16w_wide<WF, F, T, KG, GU><<<dim3(row_tiles * col_tiles * ksplit), G::NT, G::LDS_BYTES, dev->stream>>>(mats, (const char*)xh, (int)(k / 32), (int)b,
                                                                                                         row_tiles, ksplit);
  return true;
}
// Which tile.  Estimated time of a launch, us: what one chunk of a workgroup takes with a CU to itself / beside another, over the rounds of CUs, 4.6 for the
// ends, 3.7 for each round behind the first, and what pieces of k in memory cost.  Fitted to 650 timings (Q4_0, Q8_0; 77 to 1024 rows of 2048 x 2048,
// 4096 x 4096, 6144 x 4096, 4096 x 14336 and gate | up of 5632 x 2048, 14336 x 4096), 7 % off at the root mean square; the tile it chooses takes 1.9 % longer
// than the best of all on average.
struct WideTile {
  int f, t, kg;
  float alone, shared;  // shared = 0: one workgroup a CU
};
static constexpr WideTile WIDE_TILES[6] = {{4, 8, 1, 1.61f, 3.1f}, {4, 6, 1, 1.36f, 2.49f}, {2, 8, 1, 1.05f, 1.78f}, {2, 6, 1, .85f, 1.49f}, {2, 8, 2, 1.77f, 0.f}, {2, 6, 2, 1.44f, 0.f}};
// rows[0 .. nw): of the matrices; pair: gate | up, whose tiles hold rows of both and whose k stays in one workgroup (the same choice with and without the
// epilogue: the same sums); six_bits: Q6_K, whose registers hold no tile of 4 x 8; -> index into WIDE_TILES; parts: chunks' time, rounds of CUs
static int f16w_wide_tile(bool six_bits, const size_t* rows, int nw, size_t k, size_t b, bool pair, size_t n_cu, size_t ws_floats, int* ksplit, float (&parts)[2]) {
  size_t total = 0;
  for (int j = 0; j < nw; j++) total += rows[j];
  int best = -1;
  float least = 0.f;
  *ksplit = 1;
  for (int c = 0; c < 6; c++) {
    const WideTile& w = WIDE_TILES[c];
    if ((!pair && w.f == 2 && w.kg == 1) || (six_bits && c == 0)) continue;
    const size_t tile = 64 * (size_t)w.f, cols = (b + 16 * w.t - 1) / (16 * w.t);
    size_t tiles = 0;
    for (int j = 0; j < (pair ? 1 : nw); j++) tiles += pair ? (2 * rows[j] + tile - 1) / tile : (rows[j] + tile - 1) / tile;
    for (int ks = 1; ks <= (pair ? 1 : 8); ks *= 2) {
      const size_t pieces = (size_t)(ks * w.kg), chunks = (((k / 128 + pieces - 1) / pieces) + 1) & ~(size_t)1;
      if (ks > 1 && (chunks * (pieces - 1) >= k / 128 || (size_t)(ks - 1) * total * b > ws_floats)) break;
      float rounds;
      const float chunks_us = f16w_chunk_us(tiles * cols * ks, n_cu, w.alone, w.shared, &rounds) * (float)chunks;
      const float us = chunks_us + 4.6f + 3.7f * (rounds - 1.f) + (ks > 1 ? 4.f + 1.2e-6f * (float)ks * (float)(total * b) : 0.f);
      if (best < 0 || us < least) {
        best = c;
        least = us;
        *ksplit = ks;
        parts[0] = chunks_us;
        parts[1] = rounds;
      }
    }
  }
  return best;
}
// By format, against launch_gemm_f16w's own estimate (f16w_narrow_us): fitted to which of the two kernels is the faster one (there)
float f16w_wide_us(uint32_t dt, const size_t* m, int nw, size_t k, size_t b, size_t n_cu, size_t ws_floats, bool deferred) {
  size_t total = 0;
  for (int j = 0; j < nw; j++) total += m[j];
  float parts[2] = {};
  int ks = 1;
  f16w_wide_tile(dt == CRABML_HIP_Q6_K, m, nw, k, b, false, n_cu, ws_floats, &ks, parts);
  const float format = dt == CRABML_HIP_Q4_0 ? .76f : dt == CRABML_HIP_Q4_1 ? .78f : dt == CRABML_HIP_Q8_0 ? 1.31f : dt == CRABML_HIP_Q4_K ? .92f : 1.42f;
  return 4.7f + 2.5f * (parts[1] - 1.f) + format * parts[0] +
         (ks == 1 ? 0.f : deferred ? .9e-6f * (float)ks * (float)(total * b) : 3.3f + 1.5e-6f * (float)ks * (float)(total * b));
}
template <int WF>
static bool launch_wide_fmt(crabml_hip_device* dev, int tile, bool gu, F16wMats& mats, const size_t* m, int nw, size_t k, const void* xh, size_t b, int ksplit) {
  if constexpr (WF != WF_Q6_K)
    if (tile == 0)
      return gu ? launch_wide_t<WF, 4, 8, 1, true>(dev, mats, m, nw, k, xh, b, 1) : launch_wide_t<WF, 4, 8, 1, false>(dev, mats, m, nw, k, xh, b, ksplit);
  switch (tile) {
    case 1: return gu ? launch_wide_t<WF, 4, 6, 1, true>(dev, mats, m, nw, k, xh, b, 1) : launch_wide_t<WF, 4, 6, 1, false>(dev, mats, m, nw, k, xh, b, ksplit);
    case 2: return gu ? launch_wide_t<WF, 2, 8, 1, true>(dev, mats, m, nw, k, xh, b, 1) : launch_wide_t<WF, 2, 8, 1, false>(dev, mats, m, nw, k, xh, b, ksplit);
    case 3: return gu ? launch_wide_t<WF, 2, 6, 1, true>(dev, mats, m, nw, k, xh, b, 1) : launch_wide_t<WF, 2, 6, 1, false>(dev, mats, m, nw, k, xh, b, ksplit);
    case 4: return gu ? launch_wide_t<WF, 2, 8, 2, true>(dev, mats, m, nw, k, xh, b, 1) : launch_wide_t<WF, 2, 8, 2, false>(dev, mats, m, nw, k, xh, b, ksplit);
    default: return gu ? launch_wide_t<WF, 2, 6, 2, true>(dev, mats, m, nw, k, xh, b, 1) : launch_wide_t<WF, 2, 6, 2, false>(dev, mats, m, nw, k, xh, b, ksplit);
  }
}
bool launch_f16w_wide(crabml_hip_device* dev, uint32_t dt, F16wMats mats, const size_t* m, int nw, size_t k, const void* xh, size_t b, bool pair, bool gu,
                      size_t ws_floats, int* ksplit) {
  if (b <= 64 || k % 256 != 0) return false;
  for (int j = 0; j < nw; j++)
    if (m[j] * k >= (size_t)1 << 32) return false;  // (32-bit offsets into the quants)
  float parts[2];
  const bool forced = dev->wide_tile >= 0 && !(dt == CRABML_HIP_Q6_K && dev->wide_tile == 0);
  const int tile = forced ? dev->wide_tile : f16w_wide_tile(dt == CRABML_HIP_Q6_K, m, nw, k, b, pair, (size_t)dev->n_cu, ws_floats, ksplit, parts);
  switch (dt) {
    case CRABML_HIP_Q4_0: return launch_wide_fmt<WF_Q4_0>(dev, tile, gu, mats, m, nw, k, xh, b, *ksplit);
    case CRABML_HIP_Q8_0: return launch_wide_fmt<WF_Q8_0>(dev, tile, gu, mats, m, nw, k, xh, b, *ksplit);
    case CRABML_HIP_Q4_1: return launch_wide_fmt<WF_Q4_1>(dev, tile, gu, mats, m, nw, k, xh, b, *ksplit);
    case CRABML_HIP_Q4_K: return launch_wide_fmt<WF_Q4_K>(dev, tile, gu, mats, m, nw, k, xh, b, *ksplit);
    case CRABML_HIP_Q6_K: return launch_wide_fmt<WF_Q6_K>(dev, tile, gu, mats, m, nw, k, xh, b, *ksplit);
  }
  return false;
}

}  // namespace crabml_hip

extern "C" int crabml_hip_debug_wide_tile(uint32_t dtype, size_t m0, size_t m1, size_t m2, size_t k, size_t b, int32_t pair, int32_t n_cu, size_t ws_floats,
                                          int32_t* tile) {
  using namespace crabml_hip;
  if (!tile || n_cu < 1 || m0 == 0 || b <= 64 || k == 0 || k % 256 != 0) return CRABML_HIP_BAD_INPUT;
  const size_t rows[3] = {m0, m1, m2};
  float parts[2];
  const WideTile& w = WIDE_TILES[f16w_wide_tile(dtype == CRABML_HIP_Q6_K, rows, m2 ? 3 : m1 ? 2 : 1, k, b, pair != 0, (size_t)n_cu, ws_floats, tile + 3, parts)];
  tile[0] = w.f;
  tile[1] = w.t;
  tile[2] = w.kg;
  return 0;
}
