// graph_steps.hpp -- several decode steps of a greedy run behind one another in one graph: how many, and from when on
//
// A graph's two ends cost 6 to 7 us between two launches (measured with graphs of 35 and 140 small kernels), and inside one the sampler's second
// stage and the next step's embedding are one launch: eight steps of the hybrid decoder from one graph against eight, us, 4 layers of width 512
// with one row 778 -> 759, of width 2048 with one / four rows 1594 -> 1557 / 1823 -> 1784, latent and windowed layers 1928 -> 1893 / 2127 -> 2078.
// Against that stands the capture, inside the call that makes it: 1.4 to 2 us a launch (184 launches 250 to 380 us, 378 600 us, 1944 3500 us).
#pragma once
#include <algorithm>
#include <cstddef>

namespace crabml_hip {

// what a graph holds at most: a capture stays below a millisecond, and what is kept (for every batch size or attention form) is bounded
constexpr size_t GRAPH_STEPS = 8, GRAPH_NODES = 384;
constexpr double STEP_GAIN_US = 5.0, NODE_COST_US = 2.0;

// steps in a graph where one step is `nodes` launches (1: a graph of its own each)
inline int steps_a_graph(size_t nodes, size_t seq_len) {
  const size_t n = nodes ? std::min({GRAPH_STEPS + 0, GRAPH_NODES / nodes, seq_len / 2}) : 0;
  return n < 2 ? 1 : (int)n;
}
// Whether such a graph has earned its capture: `done` steps, those made one at a time so far and those that a run is about to make, would have won
// what it costs.  (A run that is long enough captures at once; shorter ones do when they have made up for it together.)
inline bool steps_graph_earned(size_t nodes, int steps, size_t done) {
  return steps > 1 && done * STEP_GAIN_US * (steps - 1) / steps >= (double)nodes * steps * NODE_COST_US;
}

}  // namespace crabml_hip
