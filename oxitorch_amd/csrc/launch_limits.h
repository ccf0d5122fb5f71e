// The largest launch. Host code without HIP headers.
#pragma once

#include <cstdint>

namespace oxi {

// HIP refuses a launch of 2^32 threads or more in one grid dimension (the
// dispatch counts threads in 32 bits) and of 2^31 blocks or more.
inline bool grid_fits(int64_t blocks, int64_t threads) {
  return blocks < ((int64_t)1 << 31) && blocks <= 0xffffffffll / threads;
}

}  // namespace oxi
