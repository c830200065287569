// gemm_f16w.hip -- the FAST prompt pass's weight GEMM, its operands, and its kernel for up to 64 rows, widths that are no multiple of 256 and launches of few
// workgroups; the others: gemm_f16w_wide.hip (crabml_hip_llama_prefill on the fast device; Q4_0 / Q8_0 weights x Q8_0 rows,
// Q4_1 x Q8_1, Q4_K / Q6_K x Q8_K): weight-stationary on the f16 matrix cores.
//
// matmul_vec with a batched rhs is `C[b, m] = W[m, k] . x[b, k]` (matmul_vec.rs:41-76: the (b, k) rhs contract; llama2.rs:111-129).
// The bit-exact form (gemm_mfma.hip: exact int8 tiles, then the reference's per-block `sumf += (sumi as f32 * d_w) * d_x`) pays
// 12-16 VALU operations per MFMA for that scaling -- it is VALU-issue-bound at 14 % MfmaUtil (profiles/r05_prefill_gemm_experiments.md).
// Here the block scales are folded into the OPERANDS and the sum runs in f32 inside the matrix core across all blocks:
//   A' = (q_w - 8) * d_w   as f16: q_w - 8 exact, ONE rounding of the product (v_pk_mul_f16)
//   B' = q_x * d_x         as f16: one rounding (k_q8_0_rows_to_f16: once per activation matrix, not per weight row tile)
//   C  = sum_k A' B'       in f32 (v_mfma_f32_16x16x32_f16), no per-block work at all.
// A deviation of the fast tier only (two extra f16 roundings per product against the reference's exact integer block dots; inside
// FAST_TOL, tests/test_hip_prefill.py); matmul_vec and the strict-order device keep the bit-exact int8 kernel.
//
// Tiling (what round 5's f16 experiment lacked): a wave owns F 16-row fragments x T = 8 column tiles of 16 prompt rows and unpacks
// each A fragment ONCE per 32 k-slots -- 15 VALU operations -- for T MFMAs: 15 F / (F T) < 2 VALU per MFMA, 0.9 with the staging
// amortized (the int8 kernel: 12 for its scaling alone).  A fragments come straight from global memory in MFMA layout: lane (i, g) loads the whole
// 16-byte block kb0 + g of row i (64 contiguous bytes per row and chunk) and step s = 0..3 of the chunk feeds dword s of every
// lane -- an MFMA's 32 k-slots then span FOUR blocks (8 elements of each), which the folded scales allow.  B' tiles (128 columns x
// 128 k-slots x 2 B = 32 KB per chunk) go through LDS, double-buffered, one barrier per chunk, shared by the workgroup's four waves;
// the fragment reads are conflict-free ds_read_b128 (layout: GemmF16Geo), a group of tiles ahead of the MFMAs that consume them.
//
// Q8_0 weights: the lane's block is 32 bytes (two loads); step s takes dwords s and 4 + s -- the same k-slot order as Q4_0's nibbles,
// so both formats share one B'.  A' = q_w * d_w (q_w exact).
// Q4_K weights (Q8_K rows): a chunk is HALF a super-block -- lane (i, g) loads the 16-byte class-major piece h of pair g (dword s =
// class 4 h + s: elements 8 k + 4 h + s of sub-blocks 2 g (low nibbles) and 2 g + 1 (high); common.hpp) and, once per super-block, the
// 16-byte header.  A' = n * fl16(d * sc) - fl16(dmin * m) (buf_q4_k.rs:225-263's d * sc * q - dmin * m, per element): n exact, the
// product exact inside ONE v_pk_fma_f16, so three f16 roundings per weight element; B' = q_x * d_x from the Q8_K planes in the
// matching slot order (k_rows_to_f16<1>).
// Q4_1 weights (Q8_1 rows): Q4_0's loads and slot order; A' = n * d + m in one v_pk_fma_f16 (buf_q4_1.rs: d * q + m per element --
// the rows' `s` term of the integer form is not needed).
// Q6_K weights (Q8_K rows): a chunk is one 128-element half of a super-block -- lane (i, g) loads 16 bytes of ql (g < 2: ql[0..31],
// the low nibbles are quarter 0, the high ones quarter 2; g >= 2: ql[32..63], quarters 1 and 3; buf_q6_k.rs:21-48) and the 16 bytes
// of qh that carry the same l's two high bits, and once per super-block the 16 int8 scales and d.  A' = (q - 32) * fl16(d * sc),
// q - 32 exact.  Its own B' slot order (k_rows_to_f16<2>): a Q4_K_M layer converts the rows once per order it needs.
#include <cstdlib>
#include <type_traits>

#include "gemm_f16w.hpp"

namespace crabml_hip {

// ---- B': the rows of a prompt pass as pre-scaled f16, in the GEMM's k-slot order: xh[col][kb][32] f16 ------------------------
// (the slot orders and the conversion of one 8-slot group: f16w_rows.hpp, shared with the row kernels that write B' themselves)
// Q8_K rows (Q4_K weights): slot group kb = 4 cc + g of chunk cc = (super-block, half h), step s = class l = 4 h + s of pair g;
// slot e: k = 0, 2, 1, 3 of sub-block 2 g (e < 4) / 2 g + 1 (e >= 4), element 8 k + l -- unpack_q4_k_f16's order
// Q6_K weights: chunk cc = (super-block, half), g, step s: element 128 half + 32 (g >> 1) + 16 (g & 1) + 4 s + k (e < 4), + 64 (e >= 4)
template <int ORDER>  // 0: Q8_0 / Q8_1 rows (block order); 1: Q8_K rows for Q4_K weights; 2: Q8_K rows for Q6_K weights
__global__ __launch_bounds__(256) void k_rows_to_f16(const char* __restrict__ planes, size_t row_stride, size_t off_d, int nb,
                                                     unsigned short* __restrict__ xh) {
  const size_t col = blockIdx.y;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;  // one thread per (block, 8-slot group)
  if (t >= nb * 4) return;
  rows_to_f16_piece<ORDER>(planes + col * row_stride, off_d, t, xh + col * (size_t)nb * 32);
}
// planes: `rows` sets of activation planes (act_layout(act_qtype, k)); the slot order is the one the weight format w_dtype reads
int gemm_f16w_order(uint32_t w_dtype) { return w_dtype == CRABML_HIP_Q4_K ? 1 : w_dtype == CRABML_HIP_Q6_K ? 2 : 0; }
bool launch_rows_to_f16(hipStream_t st, uint32_t act_qtype, uint32_t w_dtype, const void* planes, size_t rows, size_t k, void* xh) {
  if (!gemm_f16w_covers(w_dtype, act_qtype) || (act_qtype == CRABML_HIP_Q8_K && k % 256 != 0)) return false;
  const ActLayout al = act_layout(act_qtype, k);
  const int nb = (int)(k / 32);
  const dim3 grid((unsigned)((nb * 4 + 255) / 256), (unsigned)rows);
  switch (gemm_f16w_order(w_dtype)) {
    case 0: k_rows_to_f16<0><<<grid, 256, 0, st>>>((const char*)planes, al.total, al.off_d, nb, (unsigned short*)xh); break;
    case 1: k_rows_to_f16<1><<<grid, 256, 0, st>>>((const char*)planes, al.total, al.off_d, nb, (unsigned short*)xh); break;
    default: k_rows_to_f16<2><<<grid, 256, 0, st>>>((const char*)planes, al.total, al.off_d, nb, (unsigned short*)xh); break;
  }
  return true;
}

// the k pieces of a split GEMM: out[j] += part[j][0] + part[j][1] + ... in piece order (deterministic), every matrix of the launch at once
struct F16wParts {
  float* out[3];
  const float* part[3];  // matrix j's first partial; the next pieces follow pstride floats apart
  size_t end4[3];        // cumulative f32x4 counts
  size_t pstride;
  int nparts;
};
__global__ __launch_bounds__(256) void k_addn_f32(F16wParts a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.end4[2]) return;
  const int j = i < a.end4[0] ? 0 : i < a.end4[1] ? 1 : 2;
  const size_t li = i - (j == 0 ? 0 : j == 1 ? a.end4[0] : a.end4[1]);
  float* o = j == 0 ? a.out[0] : j == 1 ? a.out[1] : a.out[2];
  const float* p = j == 0 ? a.part[0] : j == 1 ? a.part[1] : a.part[2];
  f32x4 v = ((const f32x4*)o)[li];
  for (int s = 0; s < a.nparts; s++) v = v + ((const f32x4*)(p + (size_t)s * a.pstride))[li];
  ((f32x4*)o)[li] = v;
}

template <int T_, int NW = 4>
struct GemmF16Geo {
  static constexpr int T = T_, CW = 16 * T;    // column tiles per wave / prompt rows per workgroup
  static constexpr int KCH = 4;                // blocks per chunk
  // An LDS buffer is [block of the chunk g][column][80 bytes]: a column's 64 bytes of one block + 16 of padding.  ds_read_b128 is
  // serviced in four 16-lane groups that mix lanes of two k-slot groups g (MI355X_MICROARCH.md, LDS: {0-3, 12-15, 20-27}, ...) over 64
  // banks: with 80-byte columns the 16 columns of a tile sit on the 16 different 16-byte slots of the 256-byte bank row (5 i mod 16),
  // and the blocks' planes are a multiple of 256 bytes apart, so every lane group is conflict-free whichever g its lanes belong to.
  static constexpr int CSTR = 80, GSTR = CW * CSTR;
  static_assert(GSTR % 256 == 0, "block planes must be whole bank rows apart");
  static constexpr int BUF = KCH * GSTR, LDS_BYTES = 2 * BUF;
  static constexpr int B_LOADS = CW * KCH * 4 / (64 * NW);  // 16-byte pieces per thread and chunk
};

// GU (F = 2, two matrices of the same shape: ffn_gate and ffn_up): fragment 0 holds 16 rows of the FIRST matrix, fragment 1 the same
// 16 rows of the SECOND -- the workgroup owns 16 NW rows of both -- and the epilogue stores h = silu(g) * u (out[0]) instead of g and u:
// the (rows, hidden) f32 pair never makes its trip through memory (llama2.rs:620-630).  One k piece only (silu is not linear).
template <int WF, int F, int T_, bool GU = false, int NW = 4>  // F 16-row fragments x T_ 16-column tiles per wave: the workgroup's NW waves own 16 NW F consecutive weight rows
// ksplit > 1: that many workgroups per output tile, each over its piece of k, each writing its own partial buffer -- ffn_down and wo
// have few row tiles and a long serial k loop (one wave per SIMD otherwise), and a short pass has few tiles altogether
__global__ __launch_bounds__(64 * NW, 2) void k_gemm_f16w(F16wMats mats, const i32x4* __restrict__ xh, int nb, int n, int row_tiles, int ksplit) {
  using G = GemmF16Geo<T_, NW>;
  constexpr int T = G::T, KCH = G::KCH, NT = 64 * NW;
  extern __shared__ __attribute__((aligned(16))) unsigned char f16w_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg();
  const int i = lane & 15, g = lane >> 4;
  int rt, ct, ks;
  {  // XCD-aware tile order (gemm_mfma.hip): the column tiles (and k halves) of a weight row tile back to back on ONE XCD
    const int per_row = (int)gridDim.x / row_tiles, col_tiles = per_row / ksplit;
    int sub;
    if ((row_tiles & 7) == 0) {
      const int x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
      sub = j % per_row;
      rt = (j / per_row) * 8 + x;
    } else {
      rt = (int)blockIdx.x % row_tiles;
      sub = (int)blockIdx.x / row_tiles;
    }
    ct = sub % col_tiles;
    ks = sub / col_tiles;
  }
  static_assert(!GU || F == 2, "gate | up: one fragment of each matrix per wave");
  const int ti = GU ? 0 : rt < mats.tiles_end[0] ? 0 : rt < mats.tiles_end[1] ? 1 : 2;  // (uniform)
  // fragment f's matrix: the row tile's (ti), or -- GU -- matrix f
#define F16W_SEL(arr, j) ((j) == 0 ? mats.arr[0] : (j) == 1 ? mats.arr[1] : mats.arr[2])
#define F16W_PTRS(f)                                                                   \
  const int mj = GU ? (f) : ti;                                                        \
  const i32x4* __restrict__ wq = F16W_SEL(wq, mj);                                     \
  const char* __restrict__ wsc = F16W_SEL(wd, mj);                                     \
  const unsigned short* __restrict__ wd = (const unsigned short*)wsc;                  \
  const i32x4* __restrict__ wh = (const i32x4*)wsc;                                    \
  const i32x4* __restrict__ w6s = (const i32x4*)F16W_SEL(ws2, mj);                     \
  const unsigned short* __restrict__ w6d = (const unsigned short*)F16W_SEL(ws3, mj);   \
  (void)wq; (void)wd; (void)wh; (void)w6s; (void)w6d; (void)wsc
  float* __restrict__ out = ks == 0 ? (ti == 0 ? mats.out[0] : ti == 1 ? mats.out[1] : mats.out[2])
                                    : (ti == 0 ? mats.out2[0] : ti == 1 ? mats.out2[1] : mats.out2[2]) + (size_t)(ks - 1) * mats.pstride;
  const int m = ti == 0 ? mats.m[0] : ti == 1 ? mats.m[1] : mats.m[2];
  const int rt_l = rt - (ti == 0 ? 0 : ti == 1 ? mats.tiles_end[0] : mats.tiles_end[1]);
  constexpr int FSTEP = GU ? 0 : 16;  // rows between a wave's fragments
  const int r0 = (rt_l * NW + wave) * (GU ? 16 : 16 * F), c0 = ct * G::CW;
  // this workgroup's chunks: [ch_lo, ch_lo + nchunks) of the row's ceil(nb / KCH)
  // (Q4_K: an even chunk is half 0 of its super-block -- the pieces start on super-block boundaries)
  const int all_chunks = (nb + KCH - 1) / KCH;
  const int per_piece = (WF == WF_Q4_K || WF == WF_Q6_K) ? (((all_chunks + ksplit - 1) / ksplit + 1) & ~1) : (all_chunks + ksplit - 1) / ksplit;
  const int ch_lo = ks * per_piece;
  const int nchunks = all_chunks - ch_lo < per_piece ? all_chunks - ch_lo : per_piece;  // (>= 1: the launcher splits only long rows)

  // A: the lane's block (row i of fragment f, block kb0 + g) and its scale.  HBM latency is several chunk times (a chunk is ~0.4 us of
  // MFMAs and a workgroup has the SIMD almost to itself): a RING of four register sets, chunk c + 3 requested while chunk c is
  // multiplied; B' (L2-resident) two chunks ahead in two register sets.  All ring indices are compile-time (chunk loop unrolled by 4).
  constexpr int NQ = (WF == WF_Q8_0 || WF == WF_Q6_K) ? 2 : 1;  // 16-byte quant loads per fragment and chunk
  i32x4 aq[4][NQ * F];
  unsigned ad[4][F];   // Q4_0 / Q8_0: the block's scale; Q4_1: d | m << 16 (of the last block, past the row's end)
  i32x4 hq[2][F];      // Q4_K: the super-block header of ring slots (0, 1) / (2, 3), fetched with the even slot; Q6_K: the 16 scales
  unsigned hd[2][F];   // Q6_K: d
  auto fetch_a = [&](auto Jc, int ch) {
    constexpr int J = decltype(Jc)::value;
    const int cc = ch_lo + (ch < nchunks ? ch : nchunks - 1);  // (past the end: re-read the last chunk, never consumed)
    if constexpr (WF == WF_Q4_K) {
      const int nsb = nb >> 3, sb = cc >> 1, h = cc & 1;
#pragma unroll
      for (int f = 0; f < F; f++) {
        F16W_PTRS(f);
        const int row = r0 + FSTEP * f + i;
        const size_t blk = (size_t)(row < m ? row : m - 1) * nsb + sb;
        aq[J][f] = __builtin_nontemporal_load(wq + blk * 8 + 2 * g + h);
        if constexpr ((J & 1) == 0) hq[J >> 1][f] = __builtin_nontemporal_load(wh + blk);
      }
    } else if constexpr (WF == WF_Q6_K) {
      const int nsb = nb >> 3, sb = cc >> 1, half = cc & 1;
#pragma unroll
      for (int f = 0; f < F; f++) {
        F16W_PTRS(f);
        const int row = r0 + FSTEP * f + i;
        const size_t blk = (size_t)(row < m ? row : m - 1) * nsb + sb;
        aq[J][2 * f] = __builtin_nontemporal_load(wq + blk * 8 + 4 * half + g);
        aq[J][2 * f + 1] = __builtin_nontemporal_load(wh + blk * 4 + 2 * half + (g & 1));  // (wh: the qh plane, 64 bytes per super-block)
        if constexpr ((J & 1) == 0) {
          hq[J >> 1][f] = __builtin_nontemporal_load(w6s + blk);
          hd[J >> 1][f] = __builtin_nontemporal_load(w6d + blk);
        }
      }
    } else {
      const int kb = cc * KCH + g;
      const int gkb = kb < nb ? kb : nb - 1;
#pragma unroll
      for (int f = 0; f < F; f++) {
        F16W_PTRS(f);
        const int row = r0 + FSTEP * f + i;
        const size_t blk = (size_t)(row < m ? row : m - 1) * nb + gkb;
#pragma unroll
        for (int u = 0; u < NQ; u++) aq[J][NQ * f + u] = __builtin_nontemporal_load(wq + blk * NQ + u);
        if constexpr (WF == WF_Q4_1)
          ad[J][f] = __builtin_nontemporal_load((const unsigned*)wsc + blk);
        else
          ad[J][f] = __builtin_nontemporal_load(wd + blk);
      }
    }
  };
  // B': 128 columns x 256 bytes per chunk, 32 / NW pieces per thread (piece p: column p / 16, 16 bytes p % 16 of the chunk): ONE 32-bit
  // byte offset per thread, advanced by a chunk = 256 bytes per fetch (the fetches come in chunk order), against a scalar base per
  // piece -- NT / 16 columns further each (global_load ... s[base], v offset: no per-piece pointer registers).  Columns past n (a ragged
  // last tile) and the look-ahead of the last iterations read whatever follows in xh -- launch_gemm_f16w's contract keeps that
  // inside the allocation; finite or not, it meets only output columns that are never stored, zero weights, or is never consumed.
  // register sets of B' pieces in flight (one wave per SIMD: the longer look-ahead; the 32-byte-per-lane formats with two fragments:
  // one set -- B' is L2-resident and a chunk of 64 MFMAs per wave is longer than an L2 round trip)
  constexpr int NBD = (F == 1 && WF == WF_Q4_0) ? 4 : (F == 2 && (WF == WF_Q8_0 || WF == WF_Q6_K)) ? 1 : 2;
  i32x4 rb[NBD][G::B_LOADS];
  const char* xbase = (const char*)xh + ((size_t)c0 * nb + (size_t)ch_lo * KCH) * 64;  // (uniform)
  const unsigned xstep = (unsigned)(NT / 16) * (unsigned)nb * 64u;
  unsigned xoff = (unsigned)(tid >> 4) * (unsigned)nb * 64u + (unsigned)(tid & 15) * 16u;
  auto fetch_b = [&](i32x4 (&r)[G::B_LOADS], int ch) {
    (void)ch;
#pragma unroll
    for (int u = 0; u < G::B_LOADS; u++) r[u] = *(const i32x4*)(xbase + (size_t)u * xstep + xoff);
    xoff += KCH * 64;
  };
  auto commit_b = [&](const i32x4 (&r)[G::B_LOADS], int buf) {
    unsigned char* S = f16w_lds + buf * G::BUF;
#pragma unroll
    for (int u = 0; u < G::B_LOADS; u++) {
      const int p = tid + NT * u, col = p >> 4, pc = p & 15;
      *(i32x4*)(S + (pc >> 2) * G::GSTR + col * G::CSTR + (pc & 3) * 16) = r[u];
    }
  };

  f32x4 acc[F][T];
#pragma unroll
  for (int f = 0; f < F; f++)
#pragma unroll
    for (int t = 0; t < T; t++) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned magic = 0x64006400u;
  asm volatile("" : "+v"(magic));  // pinned in a VGPR (and_or_magic)

  fetch_b(rb[0], 0);
  fetch_a(std::integral_constant<int, 0>{}, 0);
  fetch_a(std::integral_constant<int, 1>{}, 1);
  fetch_a(std::integral_constant<int, 2>{}, 2);
  Q4KF16Consts cs[F];  // Q4_K: the lane's pair's constants of the current super-block (made in the even slot); Q4_1: (d, m); Q6_K: d sc
  commit_b(rb[0], 0);
  // chunk c sits in rb[c % NBD] from NBD chunks before it is committed (the fetches come in chunk order: pb advances)
#pragma unroll
  for (int c = 1; c <= NBD; c++) fetch_b(rb[c % NBD], c);
  __syncthreads();
  // chunk ch (ring slot J, LDS buffer ch & 1)
  auto chunk = [&](auto Jc, int ch) {
    constexpr int J = decltype(Jc)::value;
    fetch_a(std::integral_constant<int, (J + 3) & 3>{}, ch + 3);
    const unsigned char* S = f16w_lds + (J & 1) * G::BUF + g * G::GSTR + i * G::CSTR;
    f16x2 d2[F];
    // past the row's end: scale 0 (and m 0), the slots add nothing.  (Said here and not where the scale is requested: a choice there waits for it,
    // a memory round trip a chunk -- 1400 of 4500 cycles.  512 rows, Q4_0: wo and ffn_down 79 -> 73 us on average,
    // q | k | v 64 -> 60.)
    const unsigned there = (ch_lo + ch) * KCH + g < nb ? ~0u : 0u;
#pragma unroll
    for (int f = 0; f < F; f++) {
      if constexpr (WF == WF_Q4_K) {
        if constexpr ((J & 1) == 0) cs[f] = q4k_f16_consts(hq[J >> 1][f], g);
      } else if constexpr (WF == WF_Q6_K) {
        // the lane's two scales of a half: sc[8 half + (g & 1) + 2 (g >> 1)] (low nibbles' quarter) and 4 further (high nibbles');
        // both halves' in the even slot (the odd slot's fetch re-uses the header registers): c_* = half 0, o_* = half 1
        if constexpr ((J & 1) == 0) {
          const int sh = 8 * ((g & 1) + 2 * (g >> 1));
          const float d = h2f((unsigned short)hd[J >> 1][f]);
          _Float16 c[4];
#pragma unroll
          for (int u = 0; u < 4; u++) c[u] = (_Float16)(d * (float)(signed char)(((unsigned)hq[J >> 1][f][u] >> sh) & 0xffu));
          cs[f].c_lo = f16x2{c[0], c[0]};
          cs[f].c_hi = f16x2{c[1], c[1]};
          cs[f].o_lo = f16x2{c[2], c[2]};
          cs[f].o_hi = f16x2{c[3], c[3]};
        }
      } else if constexpr (WF == WF_Q4_1) {
        const unsigned dm = ad[J][f] & there;
        cs[f].c_lo = cs[f].c_hi = __builtin_bit_cast(f16x2, (dm & 0xffffu) | (dm << 16));
        cs[f].o_lo = cs[f].o_hi = __builtin_bit_cast(f16x2, (dm >> 16) | (dm & 0xffff0000u));
      } else {
        const unsigned d = ad[J][f] & there;
        d2[f] = __builtin_bit_cast(f16x2, d | (d << 16));
      }
    }
    // B' fragments in groups of TG tiles, two groups in registers: group q + 1 is read from LDS while group q is multiplied (left
    // to itself the compiler reads ONE fragment, waits, multiplies: 32 exposed LDS round trips per chunk with the SIMD almost to
    // itself).  The scheduling barriers keep the reads of a group ahead of the MFMAs of the previous one.
    constexpr int TG = T >= 4 ? 4 : T, NG = 4 * (T / TG);  // groups per chunk (4 steps x T / TG)
    f16x8 bq[2][TG];
    auto read_group = [&](f16x8 (&dst)[TG], int q) {
      const int s = q / (T / TG), t0 = (q % (T / TG)) * TG;
#pragma unroll
      for (int t = 0; t < TG; t++) dst[t] = *(const f16x8*)(S + (t0 + t) * 16 * G::CSTR + s * 16);
    };
    read_group(bq[0], 0);
    f16x8 a[F];
#pragma unroll
    for (int q = 0; q < NG; q++) {
      const int s = q / (T / TG), t0 = (q % (T / TG)) * TG;
      if (q + 1 < NG) read_group(bq[(q + 1) & 1], q + 1);
      if (q % (T / TG) == 0) {
#pragma unroll
        for (int f = 0; f < F; f++) {
          if constexpr (WF == WF_Q4_0) a[f] = unpack_q4_0_f16((unsigned)aq[J][f][s], d2[f], magic);
          if constexpr (WF == WF_Q8_0) a[f] = unpack_q8_0_f16((unsigned)aq[J][2 * f][s], (unsigned)aq[J][2 * f + 1][s], d2[f], magic);
          if constexpr (WF == WF_Q4_K || WF == WF_Q4_1) a[f] = unpack_q4_k_f16((unsigned)aq[J][f][s], cs[f], magic);
          if constexpr (WF == WF_Q6_K)
            a[f] = unpack_q6_k_f16((unsigned)aq[J][2 * f][s], (unsigned)aq[J][2 * f + 1][s] >> (2 * (g >> 1)), (J & 1) ? cs[f].o_lo : cs[f].c_lo,
                                   (J & 1) ? cs[f].o_hi : cs[f].c_hi, magic);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < TG; t++)
#pragma unroll
        for (int f = 0; f < F; f++) acc[f][t0 + t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[f], bq[q & 1][t], acc[f][t0 + t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    commit_b(rb[(J + 1) % NBD], (J + 1) & 1);  // chunk ch + 1 into the other buffer (read last in iteration ch - 1: behind its barrier)
    fetch_b(rb[(J + 1) % NBD], ch + 1 + NBD);  // ... and the freed register set takes chunk ch + 1 + NBD
    __syncthreads();
  };
  for (int ch = 0; ch < nchunks; ch += 4) {  // (uniform conditions: every thread takes the barrier inside a chunk or none does)
    chunk(std::integral_constant<int, 0>{}, ch);
    if (ch + 1 < nchunks) chunk(std::integral_constant<int, 1>{}, ch + 1);
    if (ch + 2 < nchunks) chunk(std::integral_constant<int, 2>{}, ch + 2);
    if (ch + 3 < nchunks) chunk(std::integral_constant<int, 3>{}, ch + 3);
  }
  // D: lane (i, g) holds rows 4 g .. 4 g + 3 of column i of every tile
  if constexpr (GU) {
    if (mats.hq.planes != nullptr) {
      // h of the workgroup's 16 NW rows x CW columns through LDS (the B' buffers are done)
      constexpr int CS = 16 * NW + 4, HB = NW / 2;  // floats per column (16-byte aligned columns, four banks apart), blocks
      static_assert((size_t)G::CW * CS * sizeof(float) <= (size_t)G::LDS_BYTES, "h fits where B' was");
      float* H = (float*)f16w_lds;
      __syncthreads();
#pragma unroll
      for (int t = 0; t < T; t++) {
        f32x4 hv;
#pragma unroll
        for (int r = 0; r < 4; r++) hv[r] = f16w_silu_mul(acc[0][t][r], acc[1][t][r], mats.exp_tab);
        *(f32x4*)(H + (16 * t + i) * CS + wave * 16 + 4 * g) = hv;
      }
      __syncthreads();
      f16w_quantize_h<HB, G::CW, CS, NT>(H, mats.hq, c0, n, rt_l * HB, m);
      return;
    }
#pragma unroll
    for (int t = 0; t < T; t++) {
      const int col = c0 + 16 * t + i;
      if (col >= n) continue;
      const int row = r0 + 4 * g;
      f32x4 hv;
#pragma unroll
      for (int r = 0; r < 4; r++) hv[r] = f16w_silu_mul(acc[0][t][r], acc[1][t][r], mats.exp_tab);
      float* o = out + (size_t)col * m + row;
      if (row + 3 < m) {
        *(f32x4*)o = hv;
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (row + r < m) o[r] = hv[r];
      }
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < T; t++) {
    const int col = c0 + 16 * t + i;
    if (col >= n) continue;
#pragma unroll
    for (int f = 0; f < F; f++) {
      const int row = r0 + 16 * f + 4 * g;
      float* o = out + (size_t)col * m + row;
      if (row + 3 < m) {
        *(f32x4*)o = acc[f][t];
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (row + r < m) o[r] = acc[f][t][r];
      }
    }
  }
}

#undef F16W_PTRS
#undef F16W_SEL

// hipFuncAttributeMaxDynamicSharedMemorySize, once per (device, kernel)
static bool f16w_raise_lds(const crabml_hip_device* dev, const void* fn, int bytes) {
  static std::mutex mu;
  static std::map<std::pair<int, const void*>, int> have;
  std::lock_guard<std::mutex> g(mu);
  int& cur = have[{dev->ordinal, fn}];
  if (bytes <= cur) return true;
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
  cur = bytes;
  return true;
}
// xh: the rows' pre-scaled f16 planes (launch_rows_to_f16) inside an allocation of gemm_f16w_xh_bytes(b, k): the kernel reads whole
// 128-column tiles and up to three chunks past the last column's end; returns false when the shape is not covered
template <int WF, int F, int T, bool GU = false, int NW = 4>
static bool launch_f16w_t(crabml_hip_device* dev, const F16wMats& mats, int row_tiles, size_t k, const void* xh, size_t b, int ksplit) {
  using G = GemmF16Geo<T, NW>;
  if (!f16w_raise_lds(dev, (const void*)k_gemm_f16w<WF, F, T, GU, NW>, G::LDS_BYTES)) {  // (80 KB of dynamic LDS: raised once per device)
    (void)hipGetLastError();
    return false;
  }
  const int col_tiles = (int)((b + G::CW - 1) / G::CW);
  k_gemm_f16w<WF, F, T, GU, NW><<<dim3(row_tiles * col_tiles * ksplit), 64 * NW, G::LDS_BYTES, dev->stream>>>(mats, (const i32x4*)xh, (int)(k / 32), (int)b,
                                                                                          row_tiles, ksplit);
  return true;
}
// (tiles of 128 or 96 columns: at most 95 more than whole tiles of 128 hold)
size_t gemm_f16w_xh_bytes(size_t rows, size_t k) { return ((rows + 127) / 128 * 128 + 96) * k * 2 + 4096; }
// the weight formats the kernel covers, and the rows' format each pairs with (CpuTensorBuf::quantize's choice: buf/api.rs:142-159)
bool gemm_f16w_covers(uint32_t w_dtype, uint32_t act_qtype) {
  if (act_qtype == CRABML_HIP_Q8_0) return w_dtype == CRABML_HIP_Q4_0 || w_dtype == CRABML_HIP_Q8_0;
  if (act_qtype == CRABML_HIP_Q8_1) return w_dtype == CRABML_HIP_Q4_1;
  return act_qtype == CRABML_HIP_Q8_K && (w_dtype == CRABML_HIP_Q4_K || w_dtype == CRABML_HIP_Q6_K);
}
// wave tile: T column tiles of 16 prompt rows -- 8 (128-row workgroup tiles) from 65 rows up; short passes (a short prompt, the ragged
// tail of a long one) take 4 / 2: the MFMAs of an empty column tile cost what a full one's do
static int f16w_col_tiles_per_wave(size_t b, int variant) { return (variant & 512) ? 4 : (variant & 16) ? 8 : b <= 32 ? 2 : b <= 64 ? 4 : 8; }
// (gate | up in one tile past 64 rows is gemm_f16w_wide.hip's where k is a multiple of 256, as it is of K-quants, but for what its launcher refuses)
template <int WF>
static bool launch_f16w_fmt(crabml_hip_device* dev, const F16wMats& mats, int row_tiles, size_t k, const void* xh, size_t b, int ksplit, int F, bool gu, int T,
                            int NW) {
  if (gu) {
    if constexpr (WF != WF_Q4_K) {
      if (T == 8) {
        if constexpr (WF != WF_Q6_K)
          if (NW == 8) return launch_f16w_t<WF, 2, 8, true, 8>(dev, mats, row_tiles, k, xh, b, 1);
        return launch_f16w_t<WF, 2, 8, true>(dev, mats, row_tiles, k, xh, b, 1);
      }
    }
    return T == 2 ? launch_f16w_t<WF, 2, 2, true>(dev, mats, row_tiles, k, xh, b, 1) : launch_f16w_t<WF, 2, 4, true>(dev, mats, row_tiles, k, xh, b, 1);
  }
  if constexpr (WF != WF_Q4_K)
    if (T == 8) return F == 2 ? launch_f16w_t<WF, 2, 8>(dev, mats, row_tiles, k, xh, b, ksplit) : launch_f16w_t<WF, 1, 8>(dev, mats, row_tiles, k, xh, b, ksplit);
  if (T == 2) return F == 2 ? launch_f16w_t<WF, 2, 2>(dev, mats, row_tiles, k, xh, b, ksplit) : launch_f16w_t<WF, 1, 2>(dev, mats, row_tiles, k, xh, b, ksplit);
  return F == 2 ? launch_f16w_t<WF, 2, 4>(dev, mats, row_tiles, k, xh, b, ksplit) : launch_f16w_t<WF, 1, 4>(dev, mats, row_tiles, k, xh, b, ksplit);
}
// gate | up in full tiles: eight waves share a B' tile, which halves what the launch reads of B' (every row tile reads all of it, a gigabyte for 512
// rows of 4096) and the staging a wave does -- one workgroup a CU, where those of four waves lie two on a CU.  It pays where the last round of CUs is
// nearly full; into a part-empty one the smaller workgroups, which then have a CU each, fit better.  A whole pass of 3 layers of width 4096, eight waves / four,
// by rounds of CUs (128-row tiles / CUs): 0.5 1.00 to 1.04, 0.67 1.00 to 1.02, 0.75 0.96 to 1.00, 0.875 0.96 to 0.99, 1.0 0.98 to 1.01, 1.25 to 1.5 1.03 to
// 1.10, 1.75 0.96 to 0.98, 2.0 0.97 to 1.01, 2.2 1.03 to 1.04, 2.6 0.97 to 0.99, 3.5 0.99 to 1.00.  Widths that are no multiple of 256, which alone come here,
// Q4_0 / Q8_0, where the rule says eight: gate | up of 8640 x 3200 0.80 0.95 / 0.97, 1.86 0.99 / 0.97; 10240 x 3200 0.94 0.98 / 0.97, 1.88 1.01 / 0.99; 7680 x 2880
// 0.94 0.99 / 1.00, 1.88 1.045 / 1.02 (the one that loses); 6400 x 1600 0.98 1.01 / 0.99; 16384 x 1600 1.0 0.98 / 0.95, 2.0 0.99 / 0.97.
static bool f16w_eight_waves(size_t tiles, size_t n_cu) {
  const size_t rounds = (tiles + n_cu - 1) / n_cu;
  return rounds == 1 ? 4 * tiles >= 3 * n_cu : 20 * tiles >= 17 * rounds * n_cu;
}
// How k_gemm_f16w would take a launch: column tiles and fragments of a wave, gate | up in one tile (pair), pieces of k
struct F16wPlan {
  int T, F, ksplit;
  bool pair;
  size_t cols, row_tiles;
};
static F16wPlan f16w_plan(uint32_t dt, const size_t* m, int nw, size_t k, size_t b, size_t n_cu, size_t ws_floats, int variant) {
  F16wPlan p{};
  size_t mtot = 0;
  for (int j = 0; j < nw; j++) mtot += m[j];
  p.T = f16w_col_tiles_per_wave(b, variant);
  // Q4_K past 64 rows, where only launches of few workgroups come here: 64 columns a tile take 0.57 to 0.9 of the time of 128 (1.13 at the worst, 1536 x 4096 of 65)
  if (dt == CRABML_HIP_Q4_K && p.T == 8) p.T = 4;
  p.cols = (b + 16 * (size_t)p.T - 1) / (16 * (size_t)p.T);
  // two fragments per wave (every B' fragment read from LDS feeds two MFMAs) when 128-row tiles still cover the chip
  p.F = ((mtot + 127) / 128) * p.cols >= n_cu ? 2 : 1;
  if ((variant & 1024) && p.F == 1 && p.T == 8 && b >= 128) {  // lab: narrow launches as two fragments x four column tiles
    p.F = 2;
    p.T = 4;
    p.cols = (b + 63) / 64;
  }
  if ((variant & 7) == 1) p.F = 2;
  if ((variant & 7) == 3) p.F = 1;
  // gate | up with the SiLU * mul epilogue (out[0] = h, out[1] untouched): when 64-row tiles of both matrices cover the chip without
  // cutting k
  p.pair = nw == 2 && m[0] == m[1] && !(variant & 64) && ((m[0] + 63) / 64) * p.cols * 2 >= n_cu * 3;
  for (int j = 0; j < nw; j++) p.row_tiles += (m[j] + 64 * p.F - 1) / (64 * p.F);
  // pieces of k: double while the launch is short of ~1.5 workgroups per CU, every piece keeps >= 4 chunks (and whole super-blocks),
  // and the partial buffers fit the scratch
  const size_t chunks = (k + 127) / 128;
  p.ksplit = 1;
  if (!(variant & 8) && k % 128 == 0)
    while (p.ksplit < 8 && p.row_tiles * p.cols * p.ksplit < n_cu * 3 / 2 && chunks % (size_t)(4 * p.ksplit) == 0 &&
           chunks / (size_t)(2 * p.ksplit) >= (size_t)((variant & 32) ? 8 : 4) && (size_t)(2 * p.ksplit - 1) * mtot * b <= ws_floats)
      p.ksplit *= 2;
  return p;
}
// gate | up whose 64-row tiles give three CUs in four something to do: in gemm_f16w_wide.hip's tiles k stays whole then, with or without the epilogue
static bool f16w_wide_pair(const size_t* m, int nw, size_t b, size_t n_cu) { return nw == 2 && m[0] == m[1] && ((m[0] + 63) / 64) * ((b + 127) / 128) * 4 >= n_cu * 3; }
// Which kernel.  gemm_f16w_wide.hip's wants whole super-blocks of k, and workgroups enough: launches of few of them are faster with the 64-row tiles of this file's
// (a layer of 256 x 768 at 128 rows, q | k | v: Q4_0 7.7 us against 6.0, Q4_K 7.9 / 4.3; 1280 x 1280 Q4_K 11.6 / 9.2, Q4_0 11.1 / 12.8; 1536 x 1536 Q4_0 11.9 /
// 10.1, Q8_0 and Q6_K alike; 3072 x 3072 Q4_0 13.0 / 11.0, at 300 rows 13.6 / 24.2).  Both are estimated: a constant, what a chunk of k takes over the rounds of
// CUs, the rounds behind the first, and pieces of k, which cost a launch to add them unless the consumer does.  Fitted to 2880 launches of five formats (q | k | v, wo,
// gate | up, ffn_down of twelve models of 256 x 768 to 4096 x 11008, 65 to 1000 rows); the kernel chosen takes 0.1 to 0.2 % longer than the faster one on
// average (26 launches more than 5 %, 1.24 times as long at the worst).  Whole passes of six layers of 256 to 2048, 65 to 1000 rows, that take every launch with
// gemm_f16w_wide.hip: up to 1.17 of the time of this file's kernel alone (256 wide), 0.92 on average by this rule and none of 400 longer by more than runs differ.
static float f16w_narrow_us(uint32_t dt, const size_t* m, int nw, size_t b, size_t k, size_t n_cu, bool deferred, const F16wPlan& p) {
  size_t total = 0;
  for (int j = 0; j < nw; j++) total += m[j];
  const bool small = p.T == 4;  // (Q4_K)
  const float alone = p.F == 1 ? (small ? .56f : .82f) : small ? 1.f : 1.37f, shared = p.F == 1 ? (small ? .95f : 1.6f) : small ? 1.63f : 2.4f;
  const float format = dt == CRABML_HIP_Q4_1 ? 1.03f : dt == CRABML_HIP_Q8_0 ? 1.12f : dt == CRABML_HIP_Q6_K ? 1.2f : 1.f;
  float rounds;
  const float chunk = f16w_chunk_us(p.row_tiles * p.cols * p.ksplit, n_cu, alone, shared, &rounds);
  return (small ? 3.3f : 4.3f) + (small ? .4f : 3.2f) * (rounds - 1.f) + format * chunk * (float)(k / 128 / p.ksplit) +
         (p.ksplit == 1 ? 0.f : deferred ? 1.1e-6f * (float)p.ksplit * (float)(total * b) : 3.9f + 1.2e-6f * (float)p.ksplit * (float)(total * b));
}
static bool f16w_takes_wide(uint32_t dt, const size_t* m, int nw, size_t k, size_t b, size_t n_cu, size_t ws_floats, bool deferred, const F16wPlan& p) {
  if (b <= 64 || k % 256 != 0) return false;
  if (p.pair || f16w_wide_pair(m, nw, b, n_cu)) return true;
  return f16w_wide_us(dt, m, nw, k, b, n_cu, ws_floats, deferred) <= f16w_narrow_us(dt, m, nw, b, k, n_cu, deferred, p);
}
// nw weight matrices (one format, the same k) against the same rhs rows: out[j] (b, m[j]) = W[j] . x
// ws (nullable), ws_floats: scratch for split launches.  When the output tiles alone leave the chip underfilled -- wo / ffn_down (few
// row tiles, a long k), any short pass -- the k range is cut into 2 / 4 / 8 pieces, one workgroup each: piece 0 writes out, the
// others their own partial buffers in ws, and k_addn_f32 adds them in piece order.  (Measured and not kept: the pieces added with
// f32 atomics onto a zeroed output -- 32.4k -> 30.1k prompt tok/s, and the sum's order would vary from run to run.)
bool launch_gemm_f16w(crabml_hip_device* dev, const crabml_hip_buf* const* w, const size_t* m, int nw, size_t k, const void* xh, size_t b,
                      float* const* out, float* ws, size_t ws_floats, const unsigned short* gu_exp_tab, int* gu_done, int* defer_parts,
                      const F16wHQuant* hq) {
  if (gu_done) *gu_done = 0;
  if (defer_parts) *defer_parts = 0;
  if (nw < 1 || nw > 3 || k % 32 != 0 || b < 16) return false;
  const uint32_t dt = w[0]->dtype;
  if (dt != CRABML_HIP_Q4_0 && dt != CRABML_HIP_Q8_0 && dt != CRABML_HIP_Q4_K && dt != CRABML_HIP_Q6_K && dt != CRABML_HIP_Q4_1) return false;
  if ((dt == CRABML_HIP_Q4_K || dt == CRABML_HIP_Q6_K) && k % 256 != 0) return false;
  for (int j = 0; j < nw; j++)
    if (w[j]->dtype != dt || m[j] % 4 != 0) return false;
  // lab hook, for the launches of this file's kernel (CRABML_HIP_TEST_HOOKS=1 CRABML_HIP_F16W=n)
  static const int variant = [] {  // 1 = two fragments, 3 = one; +8 = never split k; +16 = T = 8 always; +32 = k pieces of >= 8 chunks; +64 = no gate | up epilogue; +512 = T = 4 always; +1024 = narrow launches as <2, 4>
    const char* h = getenv("CRABML_HIP_TEST_HOOKS");
    const char* e = getenv("CRABML_HIP_F16W");
    return h && h[0] == '1' && e ? atoi(e) : 0;
  }();
  F16wMats mats{};
  F16wParts parts{};
  size_t before = 0;  // output elements of the matrices before j
  mats.exp_tab = gu_exp_tab;
  for (int j = 0; j < 3; j++) {
    const int jj = j < nw ? j : nw - 1;
    const char* wp = (const char*)w[jj]->ptr;
    mats.wq[j] = (const i32x4*)wp;
    mats.wd[j] = wp + w[jj]->wl.off_scale;
    mats.ws2[j] = wp + w[jj]->wl.off_scale + w[jj]->wl.n_blocks * 64;  // (Q6_K: ql | qh | scales | d, common.hpp)
    mats.ws3[j] = wp + w[jj]->wl.off_scale + w[jj]->wl.n_blocks * 80;
    mats.out[j] = out[jj];
    mats.out2[j] = ws + before;
    mats.m[j] = (int)m[jj];
    parts.out[j] = out[jj];
    parts.part[j] = ws + before;
    if (j < nw) before += b * m[j];
    parts.end4[j] = before / 4;
  }
  mats.pstride = parts.pstride = before;
  int ksplit = 1;
  auto finish = [&](bool gu, bool hquant) {
    if (gu) *gu_done = hquant ? 2 : 1;
    if (ksplit > 1 && defer_parts != nullptr && nw == 1) {
      *defer_parts = ksplit - 1;  // the caller's next row kernel adds the pieces (ws + s * b * m, s = 0 ..) in the same order
    } else if (ksplit > 1) {
      parts.nparts = ksplit - 1;
      k_addn_f32<<<(unsigned)((parts.end4[2] + 255) / 256), 256, 0, dev->stream>>>(parts);
    }
    return true;
  };
  if (ws == nullptr) ws_floats = 0;
  const F16wPlan plan = f16w_plan(dt, m, nw, k, b, (size_t)dev->n_cu, ws_floats, variant);
  if (f16w_takes_wide(dt, m, nw, k, b, (size_t)dev->n_cu, ws_floats, defer_parts != nullptr && nw == 1, plan) || dev->wide_tile >= 0) {
    const bool pair = f16w_wide_pair(m, nw, b, (size_t)dev->n_cu), gu = pair && gu_exp_tab != nullptr && gu_done != nullptr;
    const bool hquant = gu && hq != nullptr && hq->planes != nullptr && m[0] % 32 == 0;
    if (hquant) mats.hq = *hq;
    if (launch_f16w_wide(dev, dt, mats, m, nw, k, xh, b, pair, gu, ws_floats, &ksplit)) return finish(gu, hquant);
    mats.hq = F16wHQuant{};
  }
  const bool gu = plan.pair && gu_exp_tab != nullptr && gu_done != nullptr;
  const int T = plan.T, F = gu ? 2 : plan.F;
  // (gate | up alone.  512 rows, Q4_0 183 -> 173 us, the whole request 3973 -> 3785.  The other launches, cut in k to fill the chip with the smaller
  // tiles, do not gain: ffn_down 115 -> 108, wo 35 -> 44; four fragments a wave, one wave a SIMD, lose: 183 -> 211.)
  const int NW = gu && T == 8 && dt != CRABML_HIP_Q6_K && f16w_eight_waves((m[0] + 127) / 128 * plan.cols, (size_t)dev->n_cu) ? 8 : 4;
  const bool hquant = gu && hq != nullptr && hq->planes != nullptr && m[0] % 32 == 0;
  if (hquant) mats.hq = *hq;
  int row_tiles = 0;
  for (int j = 0; j < 3; j++) {
    if (gu)
      row_tiles = (int)((m[0] + 16 * NW - 1) / (16 * NW));
    else if (j < nw)
      row_tiles += (int)((m[j] + 64 * F - 1) / (64 * F));
    mats.tiles_end[j] = row_tiles;
  }
  ksplit = gu ? 1 : plan.ksplit;
  bool ok;
  if (dt == CRABML_HIP_Q8_0)
    ok = launch_f16w_fmt<WF_Q8_0>(dev, mats, row_tiles, k, xh, b, ksplit, F, gu, T, NW);
  else if (dt == CRABML_HIP_Q4_K)
    ok = launch_f16w_fmt<WF_Q4_K>(dev, mats, row_tiles, k, xh, b, ksplit, F, gu, T, NW);
  else if (dt == CRABML_HIP_Q6_K)
    ok = launch_f16w_fmt<WF_Q6_K>(dev, mats, row_tiles, k, xh, b, ksplit, F, gu, T, NW);
  else if (dt == CRABML_HIP_Q4_1)
    ok = launch_f16w_fmt<WF_Q4_1>(dev, mats, row_tiles, k, xh, b, ksplit, F, gu, T, NW);
  else
    ok = launch_f16w_fmt<WF_Q4_0>(dev, mats, row_tiles, k, xh, b, ksplit, F, gu, T, NW);
  return ok && finish(gu, hquant);
}

void launch_add_parts(hipStream_t st, float* out, const float* ws, size_t n, int nparts) {
  F16wParts parts{};
  parts.out[0] = out;
  parts.part[0] = const_cast<float*>(ws);
  parts.end4[0] = parts.end4[1] = parts.end4[2] = n / 4;
  parts.pstride = n;
  parts.nparts = nparts;
  k_addn_f32<<<(unsigned)((n / 4 + 255) / 256), 256, 0, st>>>(parts);
}

}  // namespace crabml_hip

extern "C" int crabml_hip_debug_gateup_waves(size_t hidden, size_t rows, int32_t n_cu, int32_t* waves) {
  if (!waves || n_cu < 1) return CRABML_HIP_BAD_INPUT;
  *waves = crabml_hip::f16w_eight_waves((hidden + 127) / 128 * ((rows + 127) / 128), (size_t)n_cu) ? 8 : 4;
  return 0;
}
extern "C" int crabml_hip_debug_prompt_gemm(uint32_t dtype, size_t m0, size_t m1, size_t m2, size_t k, size_t b, int32_t n_cu, size_t ws_floats, int32_t deferred, int32_t* wide) {
  using namespace crabml_hip;
  if (!wide || n_cu < 1 || m0 == 0 || b <= 64 || k == 0 || k % 256 != 0) return CRABML_HIP_BAD_INPUT;
  const size_t m[3] = {m0, m1, m2};
  const int nw = m2 ? 3 : m1 ? 2 : 1;
  *wide = f16w_takes_wide(dtype, m, nw, k, b, (size_t)n_cu, ws_floats, deferred != 0 && nw == 1, f16w_plan(dtype, m, nw, k, b, (size_t)n_cu, ws_floats, 0));
  return 0;
}
