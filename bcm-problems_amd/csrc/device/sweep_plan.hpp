// Host side of the sync-free sweeps: what is decided from a factor's structure
// alone (no device code).
#pragma once

#include <cstdint>

namespace bcm {

// Bound of one dependency wait of a sweep launch, in seconds. A wave may wait
// for all of the launch that comes before its row, so the bound is a time that
// no launch takes: per level 20 us and 2 us for every dependency of a row (a
// level costs 0.65 to 4 us with rows of up to 8 dependencies, one staged chunk
// of 3 more some 1 us), 0.1 us for every block and column (0.3 to 2 ns as
// measured over whole sweeps), and 4 s for what else may hold the GPU.
// levels, deps_max and blocks of both sweeps together.
inline double sweep_wait_seconds(int64_t levels, int64_t deps_max, int64_t blocks, int64_t nrhs) {
  return 4.0 + (double)levels * (20e-6 + 2e-6 * (double)deps_max) + 1e-7 * (double)blocks * (double)nrhs;
}

}  // namespace bcm
