// graph_steps.hpp -- several decode steps of a greedy run behind one another in one graph: how many, and when they are captured
//
// A graph's two ends cost 6 to 7 us between two launches (measured with graphs of 35 and 140 small kernels), and inside one the sampler's second
// stage and the next step's embedding are one launch: eight steps of the hybrid decoder from one graph against eight, us, 4 layers of width 512
// with one row 778 -> 759, of width 2048 with one / four rows 1594 -> 1557 / 1823 -> 1784, latent and windowed layers 1928 -> 1893 / 2127 -> 2078.
// Against that stands the capture, 1.4 to 2 us of the host's time a launch (184 launches 250 to 380 us, 378 600 us, 1944 3500 us).  A run captures while
// the GPU is busy with steps that it has made already, 4 us a launch and more.
#pragma once
#include <algorithm>
#include <cstddef>

namespace crabml_hip {

// what a graph holds at most: what is kept (for every batch size or attention form) is bounded, and so is the time of a capture
constexpr size_t GRAPH_STEPS = 8, GRAPH_NODES = 384;
constexpr int GRAPH_SIZES = 3;  // that many steps, half of them and a quarter

// steps in the largest graph where one step is `nodes` launches (1: a graph of its own each)
inline int steps_a_graph(size_t nodes, size_t seq_len) {
  const size_t n = nodes ? std::min({GRAPH_STEPS + 0, GRAPH_NODES / nodes, seq_len / 2}) : 0;
  return n < 2 ? 1 : (int)n;
}
// Which size comes next in a run that has made `made` steps and has `left` to make: its place (steps `top` >> place), -1 for a single step.  have, failed: bits
// by place.  A size that is not there is to be captured now: the largest for the body of a run, a smaller one for what is left of it, each behind
// steps enough to cover it.
inline int next_size(size_t left, size_t made, int top, unsigned have, unsigned failed) {
  size_t at = (size_t)top;
  for (int i = 0; i < GRAPH_SIZES && at >= 2; i++, at /= 2) {
    if (left < at || failed >> i & 1) continue;
    if (have >> i & 1 || (made > at / 2 && (i == 0 || left < 2 * at))) return i;
  }
  return -1;
}

}  // namespace crabml_hip
