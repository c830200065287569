// fused_small.hpp -- every layer of a small model's decode step in one launch
// Part of the fused decode step (included by fused.hip behind fused_ffn.hpp).
//
// What bounds it: hand-overs.  A layer of the 15M-parameter model (width 288, Q8_0) is 1 MB of weights and was five launches of 3 to 4 us each, every one
// of them dispatch, a cold first load and a drain.  Here up to 32 workgroups stay for all layers and hand rows over as 8-byte {value, epoch}
// granules (one store carries data and tag, relaxed agent scope, as in nq_epilogue).  The weights of a layer's stages are asked for before the layer's
// first gather, so that a stage is a gather, a step of integer dots and a store.  Of a layer's 11 us the five gathers are 0.9 to 1.3 us each --
// store, then a load that meets it -- and the five stages 0.9 us.
// A greedy step at 100 positions, us, five launches a layer against this: 6 layers of width 288 109 -> 81 (Q8_0), 115 -> 82 (Q4_0); 2 of 512 45.6 -> 37.1;
// 8 of 64 128 -> 88; 8 of 896 149 -> 110.  Measured and left: all workgroups on one XCD (gathers 0.3 us less, weights from one L2: 77.6, 85.4, 36.7,
// 90.4, 125.3, and 32 CUs hold one such launch only); three polls under way instead of one (92) and a sleep between polls (83 to 87); the f16
// exp table instead of its computation (0.8 us a layer); heads' q, k and v rows in the head's own workgroup (a gather less, five steps of dots more).
// 4 waves share a SIMD and a wave's instruction takes 4 cycles: a stage is bound by its instructions, so what 32 lanes can do is done by one wave.
//
// One item a workgroup and stage: 32 rows of q | k | v, a head, 32 rows of wo, 32 rows of gate and up, 32 rows of ffn_down, and one 64-unit step
// a row (small_fits).  The arithmetic is that of the five launches, term by term and in their order: k_qkv, k_attn_short, k_gemv_res_nq<DEFER>,
// k_gateup_q<DEFER>; the last ffn_down normalizes exactly, as there.  All bits are theirs.
// A granule buffer is written once a layer.  Whoever writes it again has, through the chain of gathers, waited for everything that its readers made of
// it, so one copy of each is enough.  Polls are bounded -- at half of the other launches' number and without their sleeps between, so that where the two
// kinds hold CUs that the other needs it is this one that leaves, after 0.2 s -- and raise the context's fault word, and a raised word ends the others'
// waits.  The host then runs the call again in launches per layer and stays with them (small_give_up).
#pragma once

namespace crabml_hip {

#define SMALL_WGS 32
#define SMALL_LAYERS 64
#define SMALL_POLLS (1 << 20)  // 0.17 us each
#define SMALL_FAULT 3

struct SmallLayer {
  Planes wq, wk, wv, wo, gate, up, down;
  const float *w_ffn, *w_next;  // the norms behind wo and behind ffn_down
  unsigned short *kc, *vc;
};
struct SmallStep {
  const SmallLayer* layers;
  unsigned long long *g_qkv, *g_attn, *g_x1, *g_h, *g_x2;  // [rows], [dim], [dim / 32][10], [hidden / 32][9], [dim / 32][10]
  const int* state;                                        // [1] position, [4] serial
  int* fault;
  float* x;
  signed char* q;  // the planes that the front left, and the ones for the classifier
  unsigned short* d;
  int* isum;
  const float* rope;
  const unsigned short* exp_tab;
  int L, dim, kv_dim, hd, hidden, n_heads, n_kv, seq_cap, rope_dim, npairs, polls;
  float q_scale, eps;
};
// granules of a block: eight of four quants, scale | sum, and -- x1, x2 -- the block's sum of squares
#define SMALL_XG 10
#define SMALL_HG 9

// what this wave has written to LDS is there for its other lanes
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// exp_tab[x] = f16(exp(x)) of an f16 x, as f32, computed: the table's entry was 0.8 us away, once a layer.  x hi is exact (11 + 12 bits), the rest of log2 e
// is a factor 1 + y + y^2 / 2: 1.2 ulp of f32 at most over all x (v_exp_f32 is good for one).  Where that could round to another f16 than the
// table's -- within 4 ulp of halfway between two, one value in 900 -- and outside the normal f16 range, NaN among it, the table answers:
// the same bits for all 65536 x (crabml_hip_debug_exp_of_f16).
__device__ __forceinline__ float exp_of_f16(unsigned short x, const unsigned short* __restrict__ exp_tab) {
  const float f = h2f(x), hi = 0x1.714p+0f, lo = (float)(1.44269504088896340736 - 0x1.714p+0) * 0.69314718056f;
  const float e0 = __builtin_amdgcn_exp2f(f * hi), y = f * lo;
  float e = __builtin_fmaf(e0, __builtin_fmaf(y * 0.5f, y, y), e0);
  if ((__builtin_bit_cast(unsigned, e) & 0x1fffu) - 0x0ffcu <= 8u || !(e >= 0x1p-14f && e < 65504.0f)) return h2f(exp_tab[x]);
  return h2f(f2h(e));
}
__global__ __launch_bounds__(256) void k_exp_of_f16(const unsigned short* __restrict__ exp_tab, unsigned short* __restrict__ out) {
  const unsigned x = blockIdx.x * 256 + threadIdx.x;
  out[x] = f2h(exp_of_f16((unsigned short)x, exp_tab));
}

// a pointer that every lane of the wave has read from the same place
template <class T>
__device__ __forceinline__ T* scalar_ptr(T* p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v), hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
  return (T*)((unsigned long long)hi << 32 | lo);
}

template <int FMT>
__global__ __launch_bounds__(1024) void k_small_layers(const SmallStep a) {
  using F = BlockFmt<FMT>;
  const int w = blockIdx.x;
  int tid = threadIdx.x, lane = tid & 63, wave = wave_in_wg();
  struct Act {
    i32x4 q[64];
    unsigned short d[32];
    int s[32];
  };
  __shared__ Act px, po, p1, ph;  // rhs of q | k | v, wo, gate | up, ffn_down
  __shared__ float sums[2][32];
  __shared__ __attribute__((aligned(16))) float qrow[64], hv[32], hu[32];
  __shared__ __attribute__((aligned(16))) unsigned short row_k[64], row_v[64];
  __shared__ f32x2 s_acc[8][32];
  __shared__ float s_m[8], s_l[8];
  __shared__ SmallLayer table[SMALL_LAYERS];  // (a layer's pointers are then a step away, not a trip to memory)
  const int dim = a.dim, kv_dim = a.kv_dim, hd = a.hd, nblk = dim / 32, nhb = a.hidden / 32, total = dim + 2 * kv_dim;
  const int nbd = nblk, nbh = nhb;                                // blocks of a row of dim / hidden
  const bool does_qkv = w * 32 < total, does_head = w < a.n_heads, does_x = w < nblk, does_h = w < nhb;
  if (!does_qkv && !does_head && !does_x && !does_h) return;      // (whole workgroup)
  for (int i = tid; i < a.L * (int)(sizeof(SmallLayer) / 4); i += 1024) ((unsigned*)table)[i] = ((const unsigned*)a.layers)[i];
  const int pos = a.state[1];
  const unsigned epoch0 = (unsigned)a.state[4] * (unsigned)a.L + 1u;
  bool dead = false;
  auto poll = [&](const unsigned long long* p, unsigned epoch) -> unsigned {
    unsigned long long g = ld_granule(p);
    for (int tries = 1; (unsigned)(g >> 32) != epoch && !dead; tries++) {
      if (tries >= a.polls || ((tries & 255) == 0 && __hip_atomic_load(a.fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
        dead = true;
        *a.fault = SMALL_FAULT;  // a workgroup never arrived: flagged, not hung
      }
      g = ld_granule(p);
    }
    return (unsigned)g;
  };
  auto put = [&](unsigned long long* p, unsigned v, unsigned epoch) {
    __hip_atomic_store(p, ((unsigned long long)epoch << 32) | (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  // a row of planes from its blocks' granules
  auto gather_blocks = [&](const unsigned long long* g, int n, int per, unsigned epoch, Act& to, float* sums) {
    for (int i = tid; i < n * per; i += 1024) {
      const int b = i / per, j = i - b * per;
      const unsigned v = poll(g + i, epoch);
      if (j < 8) {
        ((unsigned*)to.q)[b * 8 + j] = v;
      } else if (j == 8) {
        to.d[b] = (unsigned short)v;
        to.s[b] = (int)v >> 16;
      } else {
        sums[b] = __builtin_bit_cast(float, v);
      }
    }
  };
  auto inv_rms = [&](const float* sums, float eps) { return __builtin_amdgcn_rsqf(wave_sum_f32(lane < nblk ? sums[lane] : 0.0f) * (1.0f / (float)dim) + eps); };
  // this wave's two rows of a stage, asked for ahead
  struct Two {
    typename F::Blk r0, r1;
  };
  int r2 = wave * 2;
  // (the row's base goes through scalar registers and the lane's offset is 32 bits: 64-bit offsets of every matrix, kept over all layers, spilled)
  // Rows of up to 32 units: one in each half of the wave
  auto load = [&](const Planes& p, int row, int nb, Two& b) {
    const unsigned nu = (unsigned)(nb * F::UNITS);
    const i32x4* q = as_global(scalar_ptr(p.q)) + (unsigned)row * nu;
    const unsigned short* d = as_global(scalar_ptr(p.d)) + (unsigned)row * (unsigned)nb;
    const unsigned l = nu <= 32 ? lane & 31 : lane, u = l < nu ? l : nu - 1, r = nu <= 32 ? lane >> 5 : 0;
    const unsigned r1 = nu <= 32 ? r : 1;
    b.r0.q = q[r * nu + u];
    b.r0.d = d[r * nb + u / F::UNITS];
    b.r1.q = q[r1 * nu + u];
    b.r1.d = d[r1 * nb + u / F::UNITS];
  };
  // (wave_sum_f32's order; its upper two terms are zeros where a row has 32 lanes)
  auto dots = [&](const Two& b, const Act& x, int nb, float (&s)[2]) {
    const int nu = nb * F::UNITS, l = nu <= 32 ? lane & 31 : lane, u = l < nu ? l : nu - 1;
    const XUnit xu = F::loadx(ActQ8_0{x.q, x.d, x.s}, u);
    const float t0 = F::term(b.r0, xu), v0 = row16_sum_f32(l < nu ? 0.0f + t0 : 0.0f);
    s[0] = rl_f(v0, 0) + rl_f(v0, 16);
    s[1] = rl_f(v0, 32) + rl_f(v0, 48);
    if (nu > 32) {
      const float t1 = F::term(b.r1, xu);
      s[0] += s[1];
      s[1] = wave_sum_f32(l < nu ? 0.0f + t1 : 0.0f);
    }
  };
  // rows of q | k | v: the pair's matrix, and its rotation (the same in every layer)
  const int pair0 = w * 32 + r2;
  const bool qkv_wave = pair0 < total;
  QkvEpi qe{nullptr, nullptr, nullptr, a.rope, a.state + 1, a.q_scale, dim, kv_dim, hd, a.rope_dim, a.npairs, a.seq_cap, 1};
  const QkvPre pre = qkv_preload_nb(qe, qkv_wave ? pair0 : 0);
  const int kvh = does_head ? w / (a.n_heads / a.n_kv) : 0;
  constexpr int NW = 8, LPR = 8, RPI = 64 / LPR, RR = NW * RPI, U0 = 1, U1 = 128 / RR;  // (k_attn_short)
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const int seq = pos + 1 < a.seq_cap ? pos + 1 : a.seq_cap;

  // four lanes' quants in one word, in all four
  auto pack4 = [&](signed char q) {
    int v = (int)(unsigned char)q << ((lane & 3) * 8);
    v |= dpp_i<0xB1>(v);
    return (unsigned)(v | dpp_i<0x4E>(v));
  };
  // a block's granules: the eight words of quants from each fourth lane, scale | sum and the sum of squares from two between them
  auto put_block = [&](const QLane& o, float cs, int per, unsigned long long* g, unsigned epoch) {
    const unsigned words = pack4(o.q);
    const int j = lane & 3, at = j == 0 ? lane >> 2 : 7 + j;
    const unsigned v = j == 0 ? words : j == 1 ? (unsigned)o.d | ((unsigned)o.aux << 16) : __builtin_bit_cast(unsigned, cs);
    if (j == 0 ? lane < 32 : lane < per - 7) put(g + w * per + at, v, epoch);
  };
  // wo's and ffn_down's end (nq_epilogue, one workgroup a chunk): residual, the next norm's rhs block, the chunk's sum of squares.  hv: the rows' dots
  float res = does_x && wave == 0 ? a.x[w * 32 + (lane & 31)] : 0.f;  // the residual row, both halves of wave 0 alike, from layer to layer
  auto end_rows = [&](float wn, unsigned epoch, unsigned long long* g, bool last) {
    const float v = res = hv[lane & 31] + res;  // x = matmul_out + x (llama2.rs:266 / :636)
    hv[lane & 31] = v;
    wave_lds_fence();
    float h = -0.0f;  // (even lanes the block's first 16, odd ones the others)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const f32x4 x = *(const f32x4*)(hv + (lane & 1) * 16 + 4 * j);
#pragma unroll
      for (int i = 0; i < 4; i++) h += x[i] * x[i];
    }
    const float cs = h + dpp_f<0xB1>(h);
    if (!last) {
      put_block(quant_lane32<false>(v * wn, true), cs, SMALL_XG, g, epoch);
      return;
    }
    if (lane < 32) a.x[w * 32 + lane] = v;
    if (lane == 0) put(g + w * SMALL_XG + 9, __builtin_bit_cast(unsigned, cs), epoch);
    const float cv = lane < nblk ? __builtin_bit_cast(float, poll(g + lane * SMALL_XG + 9, epoch)) : 0.0f;
    const float rms = sqrtf((0.0f + wave_sum_f32(cv)) / (float)dim + a.eps);
    const QLane o = quant_lane32<false>((v / rms) * wn, true);
    if (lane < 32) {
      a.q[w * 32 + lane] = o.q;
      if (lane == 0) {
        a.d[w] = o.d;
        a.isum[w] = o.aux;
      }
    }
  };

  Two bq;
  const int qrow0 = !qkv_wave ? 0 : pair0 < dim ? pair0 : pair0 < dim + kv_dim ? pair0 - dim : pair0 - dim - kv_dim;
  auto load_qkv = [&](const SmallLayer& y) {
    load(!qkv_wave || pair0 < dim ? y.wq : pair0 < dim + kv_dim ? y.wk : y.wv, qrow0, nbd, bq);
  };
  const size_t kv_at = ((size_t)(qrow0 / hd) * a.seq_cap + pos) * hd + qrow0 % hd;  // (a k or v row's place in the cache)
  const int x0 = does_x ? w * 32 : 0, h0 = does_h ? w * 32 : 0;
  __syncthreads();
  load_qkv(table[0]);
  for (int l = 0; l < a.L; l++) {
    // (what is derived from these is made again in each layer: kept over all of them it spilled)
    asm volatile("" : "+v"(tid), "+v"(lane), "+s"(wave), "+s"(r2));
    const SmallLayer& y = table[l];
    const unsigned epoch = epoch0 + (unsigned)l;
    // everything of this layer that does not wait for anybody (q | k | v: since the layer before)
    Two bo, bg, bu, bd;
    const unsigned short *kb = as_global(scalar_ptr(y.kc)) + (size_t)kvh * a.seq_cap * hd, *vb = as_global(scalar_ptr(y.vc)) + (size_t)kvh * a.seq_cap * hd;
    const int rc = lane / LPR, dl = lane % LPR;
    const bool col = dl * 8 < hd;
    const int c0 = col ? dl * 8 : 0;
    const unsigned live = col ? ~0u : 0u;
    i32x4 k0[U0], v0[U0];
    // (all of it in every wave, also where it has no use for it: behind a load that not every wave makes the next wait is one for all of them)
#pragma unroll
    for (int u = 0; u < U0; u++) {
      const int row = u * RR + (wave % NW) * RPI + rc, rowc = row < a.seq_cap ? row : a.seq_cap - 1;
      k0[u] = *(const i32x4*)(kb + (unsigned)(rowc * hd + c0));
      v0[u] = *(const i32x4*)(vb + (unsigned)(rowc * hd + c0));
    }
    load(y.wo, x0 + r2, nbd, bo);
    const float wn_o = as_global(scalar_ptr(y.w_ffn))[x0 + (lane & 31)], wn_d = as_global(scalar_ptr(y.w_next))[x0 + (lane & 31)];
    load(y.gate, h0 + r2, nbd, bg);
    load(y.up, h0 + r2, nbd, bu);
    load(y.down, x0 + r2, nbh, bd);
    // ---- q | k | v
    if (does_qkv) {
      if (l == 0) {
        for (int i = tid; i < dim / 4; i += 1024) ((unsigned*)px.q)[i] = ((const unsigned*)a.q)[i];
        if (tid < nblk) {
          px.d[tid] = a.d[tid];
          px.s[tid] = a.isum[tid];
        }
      } else {
        gather_blocks(a.g_x2, nblk, SMALL_XG, epoch - 1, px, sums[0]);
      }
      __syncthreads();
      if (qkv_wave) {
        float s[2];
        dots(bq, px, nbd, s);
        if (l > 0) {
          const float ir = inv_rms(sums[0], a.eps);
          s[0] *= ir;
          s[1] *= ir;
        }
        if (lane == 0) {
          float r0 = s[0], r1 = s[1];
          if (pair0 < dim + kv_dim && pre.rot) {
            r0 = s[0] * pre.c - s[1] * pre.s;
            r1 = s[0] * pre.s + s[1] * pre.c;
          }
          unsigned g0, g1;
          if (pair0 < dim) {
            g0 = __builtin_bit_cast(unsigned, r0 * a.q_scale);
            g1 = __builtin_bit_cast(unsigned, r1 * a.q_scale);
          } else {
            g0 = f2h(r0);
            g1 = f2h(r1);
            unsigned short* o = as_global(scalar_ptr(pair0 - dim < kv_dim ? y.kc : y.vc)) + kv_at;
            o[0] = (unsigned short)g0;
            o[1] = (unsigned short)g1;
          }
          put(a.g_qkv + pair0, g0, epoch);
          put(a.g_qkv + pair0 + 1, g1, epoch);
        }
      }
      if (l + 1 < a.L) load_qkv(table[l + 1]);
    }
    // ---- attention: k_attn_short with the new position's row from LDS
    if (does_head) {
      if (tid < 3 * hd) {
        const int part = tid / hd, i = tid - part * hd;
        const unsigned v = poll(a.g_qkv + (part == 0 ? w * hd : part == 1 ? dim + kvh * hd : dim + kv_dim + kvh * hd) + i, epoch);
        if (part == 0)
          qrow[i] = h2f(f2h(__builtin_bit_cast(float, v)));
        else
          (part == 1 ? row_k : row_v)[i] = (unsigned short)v;
      }
      __syncthreads();
      if (wave < NW) {
        // (selections by mask: as conditions on values from LDS the compiler made a branch of each)
        const i32x4 q0 = *(const i32x4*)(qrow + c0), q1 = *(const i32x4*)(qrow + c0 + 4);
        float qf[8];
#pragma unroll
        for (int i = 0; i < 8; i++) qf[i] = __builtin_bit_cast(float, (unsigned)(i < 4 ? q0[i & 3] : q1[i & 3]) & live);
        const i32x4 nk = *(const i32x4*)(row_k + c0), nv = *(const i32x4*)(row_v + c0);
        float m = -FLT_MAX, s_sum = 0.f, acc[8];
#pragma unroll
        for (int i = 0; i < 8; i++) acc[i] = 0.f;
        auto take = [&](const auto& kk, const auto& vv, auto n, int row0) {
          constexpr int U = decltype(n)::value;
          float s[U], mc = -INFINITY;
#pragma unroll
          for (int u = 0; u < U; u++) {
            const int row = row0 + u * RR + rc;
            const unsigned now = row == pos ? ~0u : 0u;
            float d = 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const h2 k = __builtin_bit_cast(h2, (((unsigned)nk[i] & now) | ((unsigned)kk[u][i] & ~now)) & live);
              d = __builtin_fmaf(qf[2 * i], (float)k[0], d);
              d = __builtin_fmaf(qf[2 * i + 1], (float)k[1], d);
            }
            d = group_sum<LPR>(d);
            s[u] = row < seq ? d : -INFINITY;
            mc = fmaxf(mc, s[u]);
          }
          const float mn = fmaxf(m, wave_max_f32(mc)), alpha = __expf(m - mn);
          m = mn;
          s_sum *= alpha;
#pragma unroll
          for (int i = 0; i < 8; i++) acc[i] *= alpha;
#pragma unroll
          for (int u = 0; u < U; u++) {
            const int row = row0 + u * RR + rc;
            const unsigned now = row == pos ? ~0u : 0u, old = row < pos ? ~0u : 0u;
            const float p = __expf(s[u] - mn);
            s_sum += p;
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const h2 v = __builtin_bit_cast(h2, ((unsigned)nv[i] & now) | ((unsigned)vv[u][i] & old));
              acc[2 * i] = __builtin_fmaf(p, (float)v[0], acc[2 * i]);
              acc[2 * i + 1] = __builtin_fmaf(p, (float)v[1], acc[2 * i + 1]);
            }
          }
        };
        const int first = wave * RPI;
        if (first < seq) take(k0, v0, std::integral_constant<int, U0>{}, first);
#pragma unroll 1
        for (int r0 = U0 * RR + first; r0 < seq; r0 += U1 * RR) {
          i32x4 k1[U1], v1[U1];
#pragma unroll
          for (int u = 0; u < U1; u++) {
            const int row = r0 + u * RR + rc, rowc = row < seq ? row : seq - 1;
            k1[u] = *(const i32x4*)(kb + (unsigned)(rowc * hd + c0));
            v1[u] = *(const i32x4*)(vb + (unsigned)(rowc * hd + c0));
          }
          take(k1, v1, std::integral_constant<int, U1>{}, r0);
        }
        sum_groups<LPR>(acc);
        s_sum = sum_groups<LPR>(s_sum);
        if ((lane & 8) == 0) s_acc[wave][dl * 4 + (lane >> 5) * 2 + ((lane >> 4) & 1)] = f32x2{acc[0], acc[1]};
        if (lane == 0) {
          s_m[wave] = first < seq ? m : -INFINITY;
          s_l[wave] = s_sum;
        }
      }
      __syncthreads();
      if (wave == 0) {
        // (a wave's factor from one lane: eight exponentials in each cost as much as all of the rest)
        const float mv = s_m[lane & 7];
        float M = fmaxf(mv, dpp_f<0xB1>(mv)), Ls = 0.f;
        M = fmaxf(M, dpp_f<0x4E>(M));
        M = fmaxf(M, dpp_f<0x141>(M));
        const float ev = __expf(mv - M);
        f32x2 o = {0.f, 0.f};
#pragma unroll
        for (int v = 0; v < NW; v++) {
          const float e = rl_f(ev, v);
          const f32x2 t = s_acc[v][lane & 31];
          Ls = __builtin_fmaf(s_l[v], e, Ls);
          o[0] = __builtin_fmaf(t[0], e, o[0]);
          o[1] = __builtin_fmaf(t[1], e, o[1]);
        }
        if (tid < (hd >> 1)) {
          put(a.g_attn + w * hd + 2 * tid, __builtin_bit_cast(unsigned, o[0] / Ls), epoch);
          put(a.g_attn + w * hd + 2 * tid + 1, __builtin_bit_cast(unsigned, o[1] / Ls), epoch);
        }
      }
    }
    // ---- wo
    if (does_x) {
      if (wave * 64 < dim) {
        const QLane o = quant_lane32<false>(tid < dim ? __builtin_bit_cast(float, poll(a.g_attn + tid, epoch)) : 0.f, true);
        if (tid < dim) {
          ((signed char*)po.q)[tid] = o.q;
          if ((tid & 31) == 0) {
            po.d[tid >> 5] = o.d;
            po.s[tid >> 5] = o.aux;
          }
        }
      }
      __syncthreads();
      float s[2];
      dots(bo, po, nbd, s);
      if (lane == 0) *(f32x2*)(hv + r2) = f32x2{s[0], s[1]};
      __syncthreads();
      if (wave == 0) end_rows(wn_o, epoch, a.g_x1, false);
    }
    // ---- gate | up
    if (does_h) {
      gather_blocks(a.g_x1, nblk, SMALL_XG, epoch, p1, sums[1]);
      __syncthreads();
      float sg[2], su[2];
      dots(bg, p1, nbd, sg);
      dots(bu, p1, nbd, su);
      if (lane == 0) {
        *(f32x2*)(hv + r2) = f32x2{sg[0], sg[1]};
        *(f32x2*)(hu + r2) = f32x2{su[0], su[1]};
      }
      __syncthreads();
      if (wave == 0) {  // (a lane a row: silu_mul -- sixteen waves with two rows each take four times as long to issue it)
        const float ir = inv_rms(sums[1], 1e-5f), g = hv[lane & 31] * ir, u = hu[lane & 31] * ir;
        put_block(quant_lane32<false>((g / (1.0f + exp_of_f16(f2h(-g), a.exp_tab))) * u, true), 0.f, SMALL_HG, a.g_h, epoch);
      }
    }
    // ---- ffn_down
    if (does_x) {
      gather_blocks(a.g_h, nhb, SMALL_HG, epoch, ph, sums[1]);
      __syncthreads();
      float s[2];
      dots(bd, ph, nbh, s);
      if (lane == 0) *(f32x2*)(hv + r2) = f32x2{s[0], s[1]};
      __syncthreads();
      if (wave == 0) end_rows(wn_d, epoch, a.g_x2, l + 1 == a.L);
    }
    __syncthreads();
  }
}

// one item a workgroup and stage, one step of 64 units a row; heads past 64 columns want more registers than 16 waves leave each other
inline bool small_fits(size_t layers, size_t dim, size_t kv_dim, size_t hidden, size_t n_heads, size_t hd) {
  return layers <= SMALL_LAYERS && dim % 32 == 0 && hidden % 32 == 0 && dim + 2 * kv_dim <= 32 * SMALL_WGS && hidden <= 32 * SMALL_WGS && n_heads <= SMALL_WGS &&
         hd % 8 == 0 && hd <= 64;
}
inline int small_workers(int dim, int kv_dim, int hidden, int n_heads) {
  const int n = (dim + 2 * kv_dim + 31) / 32, m = hidden / 32;
  return n > m ? (n > n_heads ? n : n_heads) : m > n_heads ? m : n_heads;
}
inline auto small_kernel(uint32_t fmt) { return fmt == CRABML_HIP_Q8_0 ? k_small_layers<CRABML_HIP_Q8_0> : k_small_layers<CRABML_HIP_Q4_0>; }

}  // namespace crabml_hip
