// hybrid_step.hpp -- the hybrid decoder's decode step: one token of each of up to HYB_STEP_ROWS sequences, five launches per layer
//   k_gemv_bf16<RMS, ACT>         norm 1 + every projection of both mixers + their activations
//   k_mix_step                    both mixers: cache append + attention (split over cached rows, merged by the last workgroup to
//                                 finish) and the linear-attention state update, side by side in one grid
//   k_gemv_bf16<SPLIT, RESIDUAL>  both output projections (one matrix) + the linear branch's norm + residual (+ what a pass adds)
//   k_gemv_bf16<RMS, XIELU>       norm 2 + up projection + activation
//   k_gemv_bf16<PLAIN, RESIDUAL>  down projection + residual (+ what a pass adds)
// Tokens, positions and the sequences' state pointers are read from device memory, so a captured graph serves every step.
#pragma once
#include <cfloat>

#include "hybrid_common.hpp"
#include "prefetch.hpp"
#include "sampler.hpp"

namespace crabml_hip {

#define HYB_STEP_ROWS 16
#define MIX_ROWS 64  // attention workgroups share cached rows in multiples of this
#define MIX_HEADS 4  // query heads per attention workgroup
#define MIX_THREADS 512

struct StepSeq {
  int token, pos;
  char* slab;
};

// A step's front: embedding and what the first norm reads, a workgroup per row.  With pick.pv it runs behind the sampler's partials, for the tokens
// that they name (the next step's front; width 0 where that step is in another graph and brings its own): combining them (every wave for itself), advancing and embedding were three launches of one memory round trip
// each, 13.6 of the 18.4 us that a 16-row step spent outside its layers and classifier (with several steps in a graph, 16 x 154 tokens of 4 layers of
// width 2048: 20629 -> 19997 us; one sequence of 81 tokens on latent and windowed layers 12734 -> 12414).
struct RowPick {
  const float* logits = nullptr;  // [rows][ld]: n of them in place of the partials
  int n = 0, ld = 0;
  const float* pv = nullptr;  // [rows][nparts]
  const int* pi = nullptr;
  int nparts = 0, out_cap = 0;
  int* count = nullptr;  // [rows] steps done
  unsigned* out = nullptr;
};
__global__ __launch_bounds__(1024) void k_front_rows(const RowPick pick, const unsigned short* __restrict__ table, StepSeq* __restrict__ seq, int width, int ldx,
                                                     float scale, const double* __restrict__ freq, float* __restrict__ x, float* __restrict__ emb,
                                                     const float* __restrict__ add_vec, const StreamMix sm, float* __restrict__ u,
                                                     unsigned short* __restrict__ x16, const float* __restrict__ gain, float* __restrict__ xss, int ld_xss) {
  const int b = blockIdx.x, tid = threadIdx.x;
  int token = seq[b].token, pos = seq[b].pos;
  if (pick.pv) {
    float bv = -INFINITY;
    int bi = -1;
    if (pick.logits) {  // (a whole workgroup)
      __shared__ float sv[16];
      __shared__ int si[16];
      bi = argmax_row(pick.logits + (size_t)b * pick.ld, pick.n, sv, si);
    } else {
      for (int i = tid & 63; i < pick.nparts; i += 64) argmax_combine(bv, bi, pick.pv[b * pick.nparts + i], pick.pi[b * pick.nparts + i]);
      argmax_wave(bv, bi);
    }
    token = bi < 0 ? 0 : bi;
    pos++;
    __syncthreads();  // (every wave has the old position)
    if (tid == 0) {
      seq[b].token = token;
      seq[b].pos = pos;
      const int n = pick.count[b];
      const size_t at = (size_t)n * gridDim.x + b;
      if (at < (size_t)pick.out_cap) pick.out[at] = (unsigned)token;
      pick.count[b] = n + 1;
    }
  }
  constexpr int NC = 4;  // columns of a thread that are requested together
  for (int c0 = tid; c0 - tid < width; c0 += NC * 1024) {
    unsigned short e[NC];
#pragma unroll
    for (int i = 0; i < NC; i++) e[i] = table[(size_t)token * width + (c0 + i * 1024 < width ? c0 + i * 1024 : width - 1)];
#pragma unroll
    for (int i = 0; i < NC; i++) {
      const int c = c0 + i * 1024;
      const bool in = c < width;
      float r = 0.f;  // what the first norm reads
      if (in) {
        const float v = __builtin_fmaf(bf2f(e[i]), scale, position_entry(pos, c, freq));
        if (sm.n) {  // every stream starts as the embedding
          for (int t = 0; t < sm.n; t++) {
            x[t * sm.stride + (size_t)b * ldx + c] = v;
            r = __builtin_fmaf(sm.in[t], v, r);
          }
          if (!x16) u[(size_t)b * ldx + c] = r;
        } else {
          if (emb) emb[(size_t)b * ldx + c] = v;
          r = add_vec ? v + add_vec[c] : v;
          x[(size_t)b * ldx + c] = r;
        }
      }
      if (!x16) continue;
      if (in) x16[(size_t)b * ldx + c] = f2bf(gain ? r * gain[c] : r);
      const int sc = ss_columns(gridDim.x);
      float q = group_sum<8>(r * r);
      if (sc == 16) q += dpp_f<0x140>(q);
      if (in && c % sc == 0) xss[(size_t)b * ld_xss + c / sc] = q;
    }
  }
}

struct MixStep {
  AttnGeom at;
  LinGeom li;
  RunState rs;
  const StepSeq* seq = nullptr;
  const float* proj = nullptr;  // [B][ldp]
  float* cat = nullptr;         // [B][ldc]: attention columns from 0, linear columns from lin_off
  unsigned short* cat16 = nullptr;  // the same as bf16, instead (nullable)
  float* ss = nullptr;          // [B][ld_ss]: H * slices square sums of the linear branch
  int ld_ss = 0;
  float* part = nullptr;        // attention partials
  float* v_kept = nullptr;      // [B][ld_vk] values that VMIX_KEEP leaves
  int ld_vk = 0;
  unsigned* tick = nullptr;     // arrivals per (sequence, kv head, head block); the last one puts it back to zero
  int B = 0, ldp = 0, ldc = 0, lin_off = 0, splits = 0, head_blocks = 0, heads = 0;
};
// Workgroups that may share a (sequence, kv head, head block)'s rows: `per` of those in the launch, `rows` a sequence can hold.  The grid is what the
// longest sequence needs (positions live on the device), and a workgroup without rows costs its dispatch -- 16 sequences x 16 kv heads x 16
// shares: 37 us for 10 rows each -- so there are no more of them than CUs beside one per (sequence, kv head, head block).  Us a launch, shares of
// 128 rows up to capacity / this rule, 16 sequences of 10 and 300 rows: 4 kv heads x 128 20.4 / 9.5 and 35.0 / 15.9, 16 x 64 37.2 / 6.4 and
// 57.8 / 9.7; one sequence of 690 rows 12.6 / 10.4 and 8.4 / 8.9.  (Twice as many workgroups: 13.7 / 19.7 and 9.3 / 13.6 for 16 sequences.)
__host__ inline int mix_shares(int n_cu, int per, int rows) {
  const int most = (rows + MIX_ROWS - 1) / MIX_ROWS, fit = n_cu / per;
  return fit < 1 ? 1 : fit < most ? fit : most;
}
// floats of one partial: per head its V sums, the running maximum and the denominator
__host__ __device__ inline int mix_part_floats(int V) { return MIX_HEADS * (V + 2); }

__device__ __forceinline__ void cat_out(float* cat, unsigned short* cat16, size_t at, float v) {
  if (cat16)
    cat16[at] = f2bf(v);
  else
    cat[at] = v;
}

// rows of a wave's round: U requests of K and V out; with them and four heads' sums a thread holds at most 128 registers, so that two workgroups
// of 512 -- the linear branch's are as large -- share a CU
template <typename T, int CLS>
struct MixRound {
  static constexpr int LPR = CLS / 8, RPI = 64 / LPR, RR = 8 * RPI;  // lanes a row, rows of a wave's request, of one from every wave
  static constexpr int U = sizeof(T) == 2 && CLS >= 128 ? 2 : 1;
  static constexpr int ONE = CLS == 64 ? 256 : 4 * U * RR < 128 ? 4 * U * RR : 128;  // rows that stay in one workgroup
};

// One workgroup: up to MIX_HEADS query heads of one kv head over its share of the cached rows; heads up to CLS wide.  What bounds it is the
// chain position -> rows -> scores -> softmax -> sums of a cold launch, so the chain has one barrier where the heads' operands are laid out and
// one where the waves meet: a row is LPR lanes x 8 elements and a wave instruction takes 64 / LPR rows; a wave keeps K and V of its rows in
// registers, scores them for every head, takes its own maximum, and adds up p * v over its rows.  Four barriers, a wave per head's softmax and LDS
// exchanges between 256 threads before that: 13.3 -> 9.1 us a launch (one sequence, 60 rows, normed q and k), 22.1 -> 9.5 (16 sequences, 10 rows,
// linear branch beside it).  A round of 64 rows adds 1.6 us at 128 columns and 0.4 at 64, handing partial sums over 3: two rounds stay in one workgroup (four of 64
// columns, four short ones of wide heads), longer ranges are shared out evenly (one sequence of 200 rows, one workgroup / four: heads of 128
// 13.5 / 10.4 us, of 64 6.6 / 7.8).
template <typename T, int CLS>
__device__ __forceinline__ void mix_attention(const MixStep& a, int blk, float* lds) {
  using M = MixRound<T, CLS>;
  constexpr int LPR = M::LPR, RPI = M::RPI, NW = MIX_THREADS / 64, RR = M::RR, U = M::U;
  const AttnGeom& g = a.at;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg();
  const int split = blk % a.splits;
  int rest = blk / a.splits;
  const int hb = rest % a.head_blocks;
  rest /= a.head_blocks;
  const int kvh = rest % g.G, b = rest / g.G;
  const StepSeq sq = a.seq[b];
  const int hpg = g.H / g.G, h0 = kvh * hpg + hb * MIX_HEADS;
  const int nh = hpg - hb * MIX_HEADS < MIX_HEADS ? hpg - hb * MIX_HEADS : MIX_HEADS, heads = a.heads;
  const float* pr = a.proj + (size_t)b * a.ldp;
  // Everything of the projected row and the heads' parameters that this thread lays out, in one round trip beside the position's: a loop that lays out
  // what it loads waits for itself before the next one asks (what is not there reads the row's start instead, and is not used).  Us a launch, loop by loop /
  // so: one sequence of 33 to 81 rows with normed q and k 9.5 / 8.2, of 2048 with a linear branch 7.5 / 6.7, four of 700 rows 13.9 / 12.4, 16 of 90 11.8 / 10.9.
  constexpr int NQ = (MIX_HEADS * CLS + MIX_THREADS - 1) / MIX_THREADS;
  float q_new[NQ], q_gain[NQ], gate[NQ];
#pragma unroll
  for (int u = 0; u < NQ; u++) {
    const int i = tid + u * MIX_THREADS, iq = h0 * g.D + (i < nh * g.D ? i : 0), iv = i < nh * g.V ? i : 0;
    q_new[u] = pr[g.cq + iq];
    q_gain[u] = *(g.q_norm ? g.q_norm + iq : pr);
    gate[u] = pr[g.gate == GATE_ELEMENT ? g.cg + h0 * g.V + iv : g.gate == GATE_HEAD ? g.cg + h0 + iv / g.V : 0];
  }
  const int ik = kvh * g.D + (tid < g.D ? tid : 0), iv = kvh * g.V + (tid < g.V ? tid : 0), ih = h0 + (tid < nh ? tid : 0);
  const float k_new = pr[g.ck + ik], k_gain = *(g.k_norm ? g.k_norm + ik : pr), v_raw = pr[g.cv + iv];
  const float v_old = *(g.vmix == VMIX_MIX ? a.v_kept + (size_t)b * a.ld_vk + iv : pr), la = *(g.vmix == VMIX_MIX ? g.lambda : pr);
  const float amp = *(g.amp ? g.amp + ih : pr), rate = *(g.amp ? g.rate + ih : pr), sink = *(g.sink ? g.sink + ih : pr);
  float* m_s = lds;                       // [NW][MIX_HEADS] the waves' maxima
  float* l_s = m_s + NW * MIX_HEADS;      // ... and denominators
  float* hp_s = l_s + NW * MIX_HEADS;     // [3][MIX_HEADS]: penalty factor, its rate, sink; then the waves' square sums of q and k
  T* kn_s = (T*)(hp_s + 3 * MIX_HEADS + 2 * NW);  // [CLS], [CLS]: the new token's row as the cache holds it
  T* vn_s = kn_s + CLS;
  float* g_s = (float*)(vn_s + CLS);      // [heads][V]: gates
  float* q_s = g_s + heads * g.V;         // [heads][D]
  float* o_s = q_s + heads * g.D;         // [NW][heads][V]
  // the new token's row, and the rows it sees: its chunk's up to itself, or the whole ring once the window has gone round
  const int in_chunk = sq.pos % g.span, n_rows = g.window && sq.pos >= g.span ? g.span : in_chunk + 1;
  int active = 1, share = n_rows;
  if (n_rows > M::ONE) {
    const int want = (n_rows + MIX_ROWS - 1) / MIX_ROWS;
    active = want < a.splits ? want : a.splits;
    share = ((n_rows + active - 1) / active + MIX_ROWS - 1) / MIX_ROWS * MIX_ROWS;
    active = (n_rows + share - 1) / share;
  }
  if (split >= active) return;  // (whole workgroup)
  const int r0 = split * share, r1 = r0 + share < n_rows ? r0 + share : n_rows;
  T* kc = as_global((T*)(sq.slab + a.rs.k)) + (size_t)kvh * g.rows * g.D;
  T* vc = as_global((T*)(sq.slab + a.rs.v)) + (size_t)kvh * g.rows * g.V;
  const bool own_new = in_chunk >= r0 && in_chunk < r1;
  const int rc = lane / LPR, c = lane % LPR * 8;
  const bool kcol = c < g.D, vcol = c < g.V;
  Oct<T> kr[U], vr[U];
  auto fetch = [&](int base) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int row = base + u * RR + rc;
      const bool in = row < r1 && row != in_chunk;
      kr[u] = vr[u] = oct_zero<T>();
      if (in && kcol) kr[u] = oct_load(kc + (size_t)row * g.D + c);
      if (in && vcol) vr[u] = oct_load(vc + (size_t)row * g.V + c);
    }
  };
  const int first = r0 + wave * RPI;
  fetch(first);
  float q_f = g.scale, k_f = 1.f;
  if (g.q_norm) {  // (the same for the whole workgroup)
    float* red = hp_s + 3 * MIX_HEADS;
    auto squares = [&](int col, int n) {  // four requests of a thread at a time
      const float* p = pr + col;
      float s = 0.f, v[4];
      for (int i = tid; i - tid < n; i += 4 * MIX_THREADS) {
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = p[i + u * MIX_THREADS < n ? i + u * MIX_THREADS : n - 1];
#pragma unroll
        for (int u = 0; u < 4; u++) s = i + u * MIX_THREADS < n ? __builtin_fmaf(v[u], v[u], s) : s;
      }
      return wave_sum_f32(s);
    };
    float sq2 = squares(g.cq, g.H * g.D), sk2 = squares(g.ck, g.G * g.D);
    if (lane == 0) {
      red[wave] = sq2;
      red[NW + wave] = sk2;
    }
    __syncthreads();
    sq2 = sk2 = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      sq2 += red[w];
      sk2 += red[NW + w];
    }
    q_f *= 1.0f / sqrtf(sq2 / (float)g.q_mean + g.eps);
    k_f = 1.0f / sqrtf(sk2 / (float)g.k_mean + g.eps);
  }
#pragma unroll
  for (int u = 0; u < NQ; u++) {
    const int i = tid + u * MIX_THREADS;
    if (i < nh * g.D) q_s[i] = q_new[u] * (g.q_norm ? q_f * q_gain[u] : q_f);
    if (i < nh * g.V) g_s[i] = (g.gate == GATE_NONE ? 1.f : gate[u]) * g.out_scale;
  }
  if (tid < g.D) kn_s[tid] = kv_from<T>(k_new * (g.k_norm ? k_f * k_gain : 1.f));
  if (tid < g.V) vn_s[tid] = kv_from<T>(g.vmix == VMIX_MIX ? __builtin_fmaf(la, v_old, (1.0f - la) * v_raw) : v_raw);
  if (tid < nh) {
    hp_s[tid] = g.amp ? amp : 0.f;
    hp_s[MIX_HEADS + tid] = g.amp ? rate : 0.f;
    hp_s[2 * MIX_HEADS + tid] = g.sink ? sink : -INFINITY;
  }
  __syncthreads();
  if (own_new && hb == 0) {  // the new row: appended to the cache by one head block, taken from LDS by all
    if (tid < g.D) kc[(size_t)in_chunk * g.D + tid] = kn_s[tid];
    if (tid < g.V) vc[(size_t)in_chunk * g.V + tid] = vn_s[tid];
    if (g.vmix == VMIX_KEEP && tid < g.V) a.v_kept[(size_t)b * a.ld_vk + kvh * g.V + tid] = v_raw;
  }
  float m[MIX_HEADS], l[MIX_HEADS], o[MIX_HEADS][8];  // m: the same in all lanes of the wave (a row of -inf scores has weight 0)
#pragma unroll
  for (int h = 0; h < MIX_HEADS; h++) {
    m[h] = -FLT_MAX;
    l[h] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) o[h][e] = 0.f;
  }
#pragma unroll 1
  for (int base = first; base < r1; base += U * RR) {
    float kf[U][8], vf[U][8], dist[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int row = base + u * RR + rc, behind = in_chunk - row;
      if (row == in_chunk) {
        if (kcol) kr[u] = oct_load(kn_s + c);
        if (vcol) vr[u] = oct_load(vn_s + c);
      }
      oct_floats(kr[u], kf[u]);
      oct_floats(vr[u], vf[u]);
      const int back = g.window && behind < 0 ? behind + g.span : behind;
      dist[u] = (float)(back > 0 ? back : 0);
    }
    if (base + U * RR < r1) fetch(base + U * RR);  // (the next round's, while this one is worked on)
#pragma unroll
    for (int h = 0; h < MIX_HEADS; h++) {
      if (h >= nh) break;  // (uniform)
      f32x4 q0 = {0.f, 0.f, 0.f, 0.f}, q1 = q0;
      if (kcol) {
        q0 = *(const f32x4*)(q_s + h * g.D + c);
        q1 = *(const f32x4*)(q_s + h * g.D + c + 4);
      }
      float s[U], mc = -INFINITY;
#pragma unroll
      for (int u = 0; u < U; u++) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) d = __builtin_fmaf(q0[e], kf[u][e], __builtin_fmaf(q1[e], kf[u][e + 4], d));
        d = group_sum<LPR>(d);
        if (g.amp) d -= hp_s[h] * __logf(__builtin_fmaf(hp_s[MIX_HEADS + h], dist[u], 1.0f));
        s[u] = base + u * RR + rc < r1 ? d : -INFINITY;
        mc = fmaxf(mc, s[u]);
      }
      const float mn = fmaxf(m[h], wave_max_f32(mc)), alpha = __expf(m[h] - mn);
      m[h] = mn;
      l[h] *= alpha;
#pragma unroll
      for (int e = 0; e < 8; e++) o[h][e] *= alpha;
#pragma unroll
      for (int u = 0; u < U; u++) {
        const float w = __expf(s[u] - mn);
        l[h] += w;
#pragma unroll
        for (int e = 0; e < 8; e++) o[h][e] = __builtin_fmaf(w, vf[u][e], o[h][e]);
      }
    }
  }
#pragma unroll
  for (int h = 0; h < MIX_HEADS; h++) {
    if (h >= nh) break;
    sum_groups<LPR>(o[h]);
    l[h] = sum_groups<LPR>(l[h]);
    float* d = o_s + (wave * heads + h) * g.V + c + (lane >> 5) * 4;
    if (LPR == 32) {
      if (vcol) *(f32x4*)d = f32x4{o[h][0], o[h][1], o[h][2], o[h][3]};
    } else if (vcol && (LPR == 16 || (lane & 8) == 0)) {
      *(f32x2*)(d + ((lane >> 4) & 1) * 2) = f32x2{o[h][0], o[h][1]};
    }
    if (lane == 0) {
      m_s[wave * MIX_HEADS + h] = first < r1 ? m[h] : -INFINITY;
      l_s[wave * MIX_HEADS + h] = l[h];
    }
  }
  __syncthreads();
  const int slot = (b * g.G + kvh) * a.head_blocks + hb;
  const int wstr = MIX_HEADS * g.V, pf = mix_part_floats(g.V), n_out = nh * g.V;
  float* base = a.part + (size_t)slot * a.splits * pf;
  __shared__ unsigned s_last;
  auto met = [&](int i, float& M, float& L) {  // output i of the workgroup's rows: its sum, the head's maximum and denominator
    const int h = i / g.V;
    M = m_s[h];
#pragma unroll
    for (int w = 1; w < NW; w++) M = fmaxf(M, m_s[w * MIX_HEADS + h]);
    L = 0.f;
    float r = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float e = __expf(m_s[w * MIX_HEADS + h] - M);
      L = __builtin_fmaf(l_s[w * MIX_HEADS + h], e, L);
      r = __builtin_fmaf(o_s[w * heads * g.V + i], e, r);
    }
    return r;
  };
  if (active > 1) {  // partials through write-through stores; whoever arrives last merges them in row order
    float* mine = base + (size_t)split * pf;
    for (int i = tid; i < n_out; i += MIX_THREADS) {
      float M, L;
      __hip_atomic_store(mine + i, met(i, M, L), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (i % g.V == 0) {
        __hip_atomic_store(mine + wstr + 2 * (i / g.V), M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(mine + wstr + 2 * (i / g.V) + 1, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's write-through stores have been acknowledged
    __syncthreads();
    if (tid == 0) s_last = __hip_atomic_fetch_add(a.tick + slot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(active - 1);
    __syncthreads();
    if (!s_last) return;
    if (tid == 0) __hip_atomic_store(a.tick + slot, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  for (int i = tid; i < n_out; i += MIX_THREADS) {
    const int h = i / g.V;
    float m = hp_s[2 * MIX_HEADS + h], l = m == -INFINITY ? 0.f : 1.f, o = 0.f;  // the sink: a key without a value (or none)
    if (active == 1) {
      float M, L;
      const float r = met(i, M, L), mx = fmaxf(m, M), w = __expf(M - mx);
      l = __builtin_fmaf(l, __expf(m - mx), L * w);
      o = r * w;
    } else {
      for (int s0 = 0; s0 < active; s0 += 16) {
        float ps[16], ms[16], ls[16], mx = m;
#pragma unroll
        for (int s = 0; s < 16; s++) {
          const float* p = base + (size_t)(s0 + s < active ? s0 + s : s0) * pf;
          ps[s] = __hip_atomic_load(p + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ms[s] = __hip_atomic_load(p + wstr + 2 * h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ls[s] = __hip_atomic_load(p + wstr + 2 * h + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int s = 0; s < 16; s++) mx = fmaxf(mx, ms[s]);
        const float w0 = __expf(m - mx);
        m = mx;
        l *= w0;
        o *= w0;
#pragma unroll
        for (int s = 0; s < 16; s++) {
          const float w = s0 + s < active ? __expf(ms[s] - mx) : 0.f;
          l = __builtin_fmaf(ls[s], w, l);
          o = __builtin_fmaf(ps[s], w, o);
        }
      }
    }
    cat_out(a.cat, a.cat16, (size_t)b * a.ldc + h0 * g.V + i, o / l * g_s[i]);
  }
}

// one head's slice of value columns: 8 threads x 4 columns, 32 groups of key rows; 256 threads a slice
__device__ __forceinline__ void mix_linear(const MixStep& a, int blk, float* lds) {
  const LinGeom& g = a.li;
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = wave_in_wg() & 3, part = wave_in_wg() >> 2;
  const int n = a.B * g.H * g.slices, unit = blk * (MIX_THREADS / 256) + part;
  const bool used = unit < n;  // (the last workgroup's second slice may be none)
  blk = used ? unit : n - 1;
  lds += part * (2 * g.D + 32 * 36);
  const int slice = blk % g.slices, h = (blk / g.slices) % g.H, b = blk / (g.slices * g.H);
  const StepSeq sq = a.seq[b];
  float* S = as_global((float*)(sq.slab + a.rs.s)) + (size_t)h * g.D * g.V;
  const float* pr = a.proj + (size_t)b * a.ldp;
  float* k_s = lds;        // [D]
  float* q_s = k_s + g.D;  // [D]
  float* o_s = q_s + g.D;  // [32][32 + 4]
  const int c = slice * LIN_SLICE + (tid & 7) * 4, grp = tid >> 3;
  const bool live = used && c < g.V;
  const bool fresh = sq.pos == 0;  // a sequence's first token: whatever the slab holds, the state is zero
  // (what comes from the projected row is asked for ahead of the state)
  const int oc = slice * LIN_SLICE + lane, occ = h * g.V + (oc < g.V ? oc : 0), dt = h * g.D + (tid < g.D ? tid : 0);
  const float k_new = pr[g.ck + dt], q_new = pr[g.cq + dt], o_gain = g.norm[occ], o_gate = pr[g.cg + occ];
  const f32x4 v_new = *(const f32x4*)(pr + g.cv + h * g.V + (c < g.V ? c : 0));
  f32x4 s[8];  // (at most 256 key rows)
#pragma unroll
  for (int u = 0; u < 8; u++) {
    const int d = grp + u * 32;
    s[u] = live && !fresh && d < g.D ? *(const f32x4*)(S + (size_t)d * g.V + c) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (tid < g.D) {
    k_s[tid] = k_new;
    q_s[tid] = q_new;
  }
  const f32x4 v = live ? v_new : f32x4{0.f, 0.f, 0.f, 0.f};
  const float dec = g.decay[h * LIN_POW + 1];
  const float factor = o_gain * (g.out_scale * o_gate);  // the output side's, for the half-wave that will need it
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 8; u++) {
    const int d = grp + u * 32;
    if (live && d < g.D) {
      const float k = k_s[d], q = q_s[d];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        s[u][e] = __builtin_fmaf(dec, s[u][e], k * v[e]);
        o[e] = __builtin_fmaf(s[u][e], q, o[e]);
      }
      *(f32x4*)(S + (size_t)d * g.V + c) = s[u];
    }
  }
  *(f32x4*)(o_s + grp * 36 + (tid & 7) * 4) = o;
  __syncthreads();
  if (wave == 0) {  // 32 columns; the upper half-wave adds nothing to the square sum
    float r = 0.f;
    if (lane < LIN_SLICE) {
#pragma unroll
      for (int i = 0; i < 32; i++) r += o_s[i * 36 + lane];
    }
    const bool in = used && lane < LIN_SLICE && oc < g.V;
    const float ss = wave_sum_f32(in ? r * r : 0.f);
    if (used && lane == 0) a.ss[(size_t)b * a.ld_ss + h * g.slices + slice] = ss;
    if (in) cat_out(a.cat, a.cat16, (size_t)b * a.ldc + a.lin_off + occ, r * factor);
  }
}

// used: workgroups of the two branches (PF: the others prefetch)
template <typename T, int CLS, bool PF>
__global__ __launch_bounds__(MIX_THREADS, 4) void k_mix_step(const MixStep a, int used, const typename PrefetchArg<PF>::type pf) {
  extern __shared__ __attribute__((aligned(16))) float mix_lds[];
  if constexpr (PF) {
    if ((int)blockIdx.x >= used) {
      prefetch_wg(pf, blockIdx.x, used, gridDim.x);
      return;
    }
  }
  const int n_attn = a.at.H ? a.B * a.at.G * a.head_blocks * a.splits : 0;
  if ((int)blockIdx.x < n_attn)
    mix_attention<T, CLS>(a, blockIdx.x, mix_lds);
  else
    mix_linear(a, blockIdx.x - n_attn, mix_lds);
}
template <typename T, int CLS>
inline void launch_mix_step_t(hipStream_t st, crabml_hip_device::ProfRec* rec, MixStep a, const PrefetchPlan& pf, int spare) {
  constexpr int NW = MIX_THREADS / 64;
  const int hpg = a.at.H ? a.at.H / a.at.G : 0;
  a.heads = hpg < MIX_HEADS ? hpg : MIX_HEADS;
  const size_t at = a.at.H ? (2 * NW + 3) * MIX_HEADS + 2 * NW + 2 * CLS * sizeof(T) / 4 + (size_t)a.heads * (a.at.D + (NW + 1) * a.at.V) : 0;
  const size_t li = a.li.H ? (size_t)(2 * a.li.D + 32 * 36) * (MIX_THREADS / 256) : 0;
  const int units = a.B * a.li.H * a.li.slices;
  const int used = (a.at.H ? a.B * a.at.G * a.head_blocks * a.splits : 0) + (units + MIX_THREADS / 256 - 1) / (MIX_THREADS / 256);
  const size_t lds = (at > li ? at : li) * sizeof(float);  // (at most 43 KiB)
  if (pf.n)
    launch_k(st, rec, k_mix_step<T, CLS, true>, dim3((unsigned)(used + spare)), dim3(MIX_THREADS), lds, a, used, pf);
  else
    launch_k(st, rec, k_mix_step<T, CLS, false>, dim3((unsigned)used), dim3(MIX_THREADS), lds, a, used, NoPrefetch{});
}
template <typename T>
inline void launch_mix_step(hipStream_t st, crabml_hip_device::ProfRec* rec, const MixStep& a, const PrefetchPlan& pf, int spare) {
  const int w = a.at.D > a.at.V ? a.at.D : a.at.V;
  if (w <= 64)
    launch_mix_step_t<T, 64>(st, rec, a, pf, spare);
  else if (w <= 128)
    launch_mix_step_t<T, 128>(st, rec, a, pf, spare);
  else
    launch_mix_step_t<T, 256>(st, rec, a, pf, spare);
}

}  // namespace crabml_hip
