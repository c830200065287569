// prefetch.hpp -- the next launch's weights into the L2 they will be read through, by workgroups of a launch that leaves memory idle
//
// A step's attention (k_attn, k_attn_s, k_attn_short) and mixers (k_mix_step) are chains of a few dependent round trips in a few workgroups.  Spare
// workgroups of those launches touch every 128-byte line of the next linear's weights (one dword a lane: 64 lines a wave instruction, no register traffic).
// Workgroup i of a launch runs on XCD i mod 8 and each XCD has an L2 of its own (4 MB), so a line helps most where the workgroup that will
// read it runs: a plan lists the consumer's workgroups with the bytes each reads, and a spare workgroup takes those of its own XCD.
// A cold launch that reads 8 / 16 / 32 MB takes 3.1 / 4.5 / 6.7 us, behind such a launch 1.7 / 2.0 / 2.7, and 2.6 / 3.8 / 5.9 where the lines
// were touched from another XCD (they are in the Infinity Cache then).  Above what the L2s hold there is nothing to win: lines are gone before they
// are read, and the launch that hosts the traffic is the longer for it.  A run of steps of the hybrid decoder with 3 / 8 / 16 rows, with / without:
// w_o of 16 MB 1.01 / 0.97 / 1.00, 32 MB 1.01 / 0.98 / 1.00, 48 MB 1.02 / 1.00 / 1.02, 64 MB 1.04 / 1.05 / 1.03, 96 MB 1.07 / 1.07 / 1.08, 128 MB 1.13 / 1.14 /
// 1.15.  No result depends on it, nor on where a workgroup runs.
#pragma once
#include "devutil.hpp"

namespace crabml_hip {

struct PrefetchPlan {
  static constexpr int MAX = 2;
  const char* p[MAX];       // workgroup first + i of the next launch (i < count) reads `bytes` bytes at p + i * bytes
  unsigned bytes[MAX];
  int first[MAX], count[MAX];
  int n;
};
// a kernel that hosts it is a template of PF, so that where there is nothing to prefetch it is the kernel without (its larger arguments alone cost a one-row step 1 %)
struct NoPrefetch {};
template <bool PF>
struct PrefetchArg {
  typedef NoPrefetch type;
};
template <>
struct PrefetchArg<true> {
  typedef PrefetchPlan type;
};
inline void prefetch_add(PrefetchPlan& pf, const void* p, size_t bytes, int first, int count) {
  if (pf.n == PrefetchPlan::MAX || bytes < 4 || count < 1) return;
  pf.p[pf.n] = (const char*)p;
  pf.bytes[pf.n] = (unsigned)bytes;
  pf.first[pf.n] = first;
  pf.count[pf.n++] = count;
}
constexpr size_t PREFETCH_MOST = (size_t)32 << 20;  // what the L2s hold
// Models whose steps read more than this (PREFETCH_MODEL behind k_attn_short; the hybrid decoder PREFETCH_MODEL_HYBRID) do without: the short hosts take
// longer than the linear gains, probably because every XCD touches pages all over a matrix and from some 4 GB of weights on their addresses are not at hand
// (32 layers of the 8B shape, 4.2 GB: attention 4.6 -> 5.9 us, wo 5.6 -> 4.6, a token 1257 -> 1285).  k_attn and k_attn_s take long enough to hide it: the
// strict device at the same 32 layers 652 tokens/s without, 668 with.  A token with / without: 8B shape in Q4_0, 1.3 GB 0.987,
// 2.3 GB 0.983, 3.2 GB 0.985, 4.2 GB 1.031; in Q8_0, 3.3 GB 0.991, 4.3 GB 1.019, 6.1 GB 1.025; width 3072, 1.8 GB 0.974.  Hybrid decoder of width 2048, 3 / 8 / 16
// rows: 0.65 GB 1.01 / 0.97 / 0.99, 1.2 GB 1.01 / 0.97 / 1.01, 2.2 GB 1.03 / 1.00 / 1.03, 4.3 GB 1.05 / 1.00 / 1.00, of width 4096, 4.2 GB 1.04 / 1.04 / 1.04.
constexpr size_t PREFETCH_MODEL = (size_t)3584 << 20, PREFETCH_MODEL_HYBRID = (size_t)1536 << 20;
// a matrix of which the next launch's workgroups take `rows` of the m rows each: row_bytes a row from p, and row_bytes2 from p2 (scales; 0: none)
inline PrefetchPlan prefetch_matrix(size_t model_bytes, size_t model_most, int m, int rows, const void* p, size_t row_bytes, const void* p2, size_t row_bytes2) {
  PrefetchPlan pf{};
  if (model_bytes > model_most || (size_t)m * (row_bytes + row_bytes2) > PREFETCH_MOST) return pf;
  prefetch_add(pf, p, row_bytes * rows, 0, m / rows);
  prefetch_add(pf, p2, row_bytes2 * rows, 0, m / rows);
  return pf;
}

// wg: this workgroup's place in the launch (x fastest); the launch's spare ones are [base, all)
__device__ __forceinline__ void prefetch_wg(const PrefetchPlan& pf, int wg, int base, int all) {
  const int x = wg & 7, at = base + ((x - base) & 7), nw = blockDim.x >> 6, lane = threadIdx.x & 63;
  const int waves = ((all - 1 - at) / 8 + 1) * nw, me = ((wg - at) >> 3) * nw + wave_in_wg();  // of this XCD
  for (int s = 0; s < pf.n; s++) {
    const char* p = pf.p[s];
    const unsigned bytes = pf.bytes[s], pieces = (bytes + 8191) >> 13;
    const int i0 = (x - pf.first[s]) & 7;
    const unsigned items = pf.count[s] > i0 ? (unsigned)((pf.count[s] - i0 + 7) >> 3) * pieces : 0;
    for (unsigned j = me; j < items; j += 2 * waves) {
      unsigned v[2];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const unsigned k = j + u * waves < items ? j + u * waves : j, i = k / pieces;
        unsigned o = (k - i * pieces) * 8192 + lane * 128;
        o = o < bytes - 3 ? o : bytes - 4;  // (the workgroup's last bytes: a line that is read anyway)
        v[u] = *as_global((const unsigned*)((size_t)(p + (size_t)(i0 + 8 * i) * bytes + o) & ~(size_t)3));
      }
      asm volatile("" ::"v"(v[0]), "v"(v[1]));  // (the loads stay; nothing is stored)
    }
  }
}

}  // namespace crabml_hip
