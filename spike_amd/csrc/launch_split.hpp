// launch_split.hpp -- host rules of how a launch's work is cut (no device code).
#pragma once
#include <stdint.h>

#include <algorithm>

namespace spk {

// Wavefronts that share a spiking unit's row in k_deliver: one per 64 synapses of the longest
// row, at most 64.  The kernel counts the tasks (spike, wavefront of its row) of up to 64
// sub-steps in 32 bits; fewer wavefronts take a row when every unit could spike in every one of
// them (5e5 units with rows of 4096 synapses and groups of 64 steps would reach 2^31).
inline int deliver_row_waves(int64_t max_row, int64_t units, int G) {
  const int64_t spikes = std::max<int64_t>(1, units * std::min(G, 64));
  const int64_t most = std::max<int64_t>(1, ((int64_t)1 << 30) / spikes);
  return (int)std::min<int64_t>(std::min<int64_t>(64, most), std::max<int64_t>(1, (max_row + 63) / 64));
}

}  // namespace spk
