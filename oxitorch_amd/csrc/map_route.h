// Which tiles a transposed elementwise launch takes. Host code without HIP
// headers.
#pragma once

#include <algorithm>
#include <cstdint>

#include "oxihip.h"

namespace oxi {

// How long an operation on one element takes.
enum OpLength { OP_SHORT, OP_LONG, OP_POW };
constexpr OpLength unary_length(int op) {
  return op == OXI_UNARY_SQRT || op == OXI_UNARY_RSQRT || op == OXI_UNARY_EXP || op == OXI_UNARY_LOG ||
                 op == OXI_UNARY_LOG2 || op == OXI_UNARY_LOG10 || op == OXI_UNARY_SIN || op == OXI_UNARY_COS ||
                 op == OXI_UNARY_TANH || op == OXI_UNARY_SIGMOID
             ? OP_LONG
             : OP_SHORT;
}
constexpr OpLength binary_length(int op) { return op == OXI_BINARY_POW ? OP_POW : OP_SHORT; }

// Whether operands of odd extents J (the inputs' unit-stride dim) x D (the
// output's) go through 64x64 LDS tiles, `blocks` of them, instead of a wave's
// registers. There a lane works its 4x4 block off serially, 16 operations even
// where the extents leave few lanes to a wave, and repeats up to 3 rows and
// columns; an LDS tile gives each thread one of the few elements, but takes a
// block for them. So long operations on tiny extents go through LDS while its
// blocks find the chip empty: tanh-GELU's VJP of (100, 7, 7) 5.4 us against
// 9.7, of (1000, 15, 5) 7.3 against 10.4, but of (2000, 7, 7) 10.3 against 7.2;
// with more lanes at work only the first of them: tanh of (140, 11, 11) 5.6
// against 7.1, of (1000, 11, 11) 6.3 against 5.2. pow, the longest: (100, 7, 7)
// 6.5 against 24, (10000, 4, 11) 42 against 44, (100, 5, 1001) 14 against 17,
// (1000, 5, 1001) 129 against 105, (1000, 12, 13) 9.0 against 8.6, (1500, 12,
// 13) 12.9 against 11.2. Short operations take registers at any size.
inline bool map_through_lds(OpLength op, int64_t J, int64_t D, int64_t blocks, int cus) {
  if (op == OP_SHORT) return false;
  // lanes of a wave that have a block
  const int64_t lanes = ((std::min<int64_t>(J, 32) + 3) / 4) * ((std::min<int64_t>(D, 32) + 3) / 4);
  if (op == OP_POW) return blocks <= (lanes <= 8 ? 40 : J <= 8 ? 8 : J <= 20 ? 4 : 0) * (int64_t)cus;
  return lanes <= 8 ? blocks <= 4 * (int64_t)cus : lanes <= 12 && blocks <= cus + cus / 2;
}

}  // namespace oxi
