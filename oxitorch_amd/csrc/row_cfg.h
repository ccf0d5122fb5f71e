// Which register-row configuration a row-wise launch takes. Host code without
// HIP headers.
#pragma once

#include <cstdint>

#include "launch_limits.h"

namespace oxi {

// Threads per block of a row kernel whose rows take TPR threads: 256 (several
// rows per block) when TPR divides 256, else one row per block of TPR.
constexpr int row_block_threads(int tpr) { return (256 % tpr == 0) ? 256 : tpr; }

// (TPR, NV) for rows of h4 float4s, encoded TPR*10 + NV; 0 when the row does
// not fit in registers. Rows keep several float4s per lane: measured on
// MI355X, one float4 per lane (192 threads per 768-float row, 1024 per
// 4096-float row) made the layer-norm forward 30% slower, the block-wide
// reductions over many waves costing more than the access pattern gains;
// 512 x 2 for a 4096-float row measured the same as 256 x 4 (layer-norm
// forward at (16384, 4096): 88.8-89.5 us against 87.7-89.3 us).
inline int pick_row_cfg(int64_t h4) {
  if (h4 <= 64) return 641;
  if (h4 <= 128) return 642;
  if (h4 <= 192) return 643;
  if (h4 <= 256) return 644;
  if (h4 <= 512) return 2562;
  if (h4 <= 1024) return 2564;
  if (h4 <= 2048) return 2568;
  return 0;
}

// The configuration of a norm's forward over `rows` rows of H floats, which
// may lie anywhere: as above by the row's float4s, rows of up to 16384 floats
// on 1024 threads of 4 (layer norm of (2048, 12288) 41 us against 74 re-reading
// the row); 0, the loop kernel of 256 threads a row, for rows of fewer than 4
// floats, longer ones, and more of them than a grid of 1024-thread blocks holds.
inline int norm_fwd_cfg(int64_t rows, int64_t H) {
  const int64_t h4 = (H + 3) / 4;
  if (H < 4) return 0;
  const int cfg = pick_row_cfg(h4);
  return cfg ? cfg : h4 <= 4096 && grid_fits(rows, 1024) ? 10244 : 0;
}

}  // namespace oxi
