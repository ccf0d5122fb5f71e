// The launch of the middle-dim softmax kernels. Host code without HIP headers.
#pragma once

#include <algorithm>
#include <cstdint>

#include "launch_limits.h"

namespace oxi {

// NT threads, TX units by TY positions a block (TX * TY = NT), NV positions a
// thread (0: streamed).
struct MidShape {
  int nt, tx, ty, nv;
  int64_t units, total, blocks;
};

inline MidShape mid_shape(int64_t outer, int64_t len, int64_t inner) {
  MidShape m;
  const int w = inner >= 4 ? 4 : 1;
  const int nv = w == 4 ? 8 : 16;  // positions a thread holds at most
  m.units = (inner + w - 1) / w;
  m.total = outer * m.units;
  m.nt = len <= 32 * nv ? 256 : 1024;
  m.ty = 1;
  while ((int64_t)m.ty * nv < len && m.ty < m.nt / 8) m.ty <<= 1;
  m.tx = m.nt / m.ty;
  const int64_t per = (len + m.ty - 1) / m.ty;
  m.nv = per <= nv / 4 ? nv / 4 : per <= nv ? nv : 0;
  m.blocks = (m.total + m.tx - 1) / m.tx;
  return m;
}

// Outer indices a launch: its grid stays below the thread limit (several
// threads walk a column, so 2^31 columns of 17 positions, 146 GB, do not fit one).
inline int64_t mid_outer_max(int64_t len, int64_t inner) {
  const MidShape m = mid_shape(1, len, inner);
  const int64_t blocks = 0xffffffffll / m.nt;  // a block count that grid_fits
  return std::max<int64_t>(1, blocks * m.tx / m.units);
}

}  // namespace oxi
