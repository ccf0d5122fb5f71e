// Which launch a dim reduction takes: the plan of its strides and the rules
// over sizes, strides and alignment. Host code without HIP headers.
#pragma once

#include <algorithm>
#include <cstdint>

#include "launch_limits.h"
#include "oxihip.h"

namespace oxi {

struct RPlan {
  int nd;                      // dims other than the reduced one
  int64_t size[OXI_MAX_DIMS];  // row-major order of the remaining dims
  int64_t st[OXI_MAX_DIMS];
  int64_t len;                 // reduced dim size
  int64_t rst;                 // reduced dim stride
};

// Where the launch shapes change, with times on MI355X (before: one wave per
// contiguous strip reading single floats, one thread per output or four).
// Contiguous strips of up to WAVE_MAX_LEN floats take a wave each (mean over
// (16384, 768) 16.3 -> 8.9 us), longer ones a block of 256 threads, or 1024
// while there are under two strips per CU: argmax over (4096, 50257) 438 ->
// 128 us, sum over (64, 16384) 31.6 -> 4.3 us.
constexpr int64_t WAVE_MAX_LEN = 2048;
// Those of up to WAVE_SHORT_LEN read single floats, as float4s half the lanes
// and more would have nothing to do: sums over (524288, 32) 77 us against 98,
// (262144, 64) 40.5 against 50, (131072, 128) 25.1 against 26.0, but (83886,
// 200) 23.8 against 19.0.
constexpr int64_t WAVE_SHORT_LEN = 128;
// From SPLIT_MIN_LEN on, and with fewer strips than CUs, the strips are cut
// into parts of a multiple of SPLIT_MIN_PART floats (four float4s a thread),
// about SPLIT_BLOCKS_PER_CU a CU in all: the norm of 12.6M values 46
// ms -> 14 us of kernels (3.6 TB/s) with the input in the Infinity Cache (72
// ms before from HBM), 1M values 1510 -> 10 us a call. The second launch takes
// about 5 us, what one block takes for 50000 floats more.
constexpr int64_t SPLIT_MIN_LEN = 65536;
constexpr int64_t SPLIT_BLOCKS_PER_CU = 4;
constexpr int64_t SPLIT_MIN_PART = 4096;
constexpr int64_t SPLIT_MAX_PARTS = 1024;  // in a strip (LDS holds their states in a captured launch)
// Strided strips of COLS_MIN_LEN positions or more, of up to COLS_MAX_OUT
// outputs, go through LDS: the column sums of (16384, 768) 760-1200 -> 59 us, of
// (1024, 16384) 68 -> 25 us, of (4096, 8000) 298 -> 42 us, the maxima of
// (16384, 768) 760-1200 -> 38 us. With more outputs a thread per output fills the
// chip: (512, 65536) 22 us there against 57 through LDS. Two and four
// stages of loads in flight instead of one: 61-90 us at (16384, 768), the
// staging then holding up the fold.
constexpr int64_t COLS_MIN_LEN = 64;
constexpr int64_t COLS_MAX_OUT = 16384;
constexpr int COLS_C = 16;             // adjacent outputs a block takes there
constexpr int COLS_THREADS = 512 + 64;  // its loading threads and the wave that folds
// A block stages 512 positions of 16 columns whatever it needs of them, and
// its 66 KB of LDS let two run on a CU (a round of blocks): outputs that do not
// lie side by side make many blocks. Past one round the strips are this long
// per round, else a thread per output is faster: sums over dim 1 of (8192, 64, 2)
// (16 rounds) 9.7 us there against 54 through LDS, of (4096, 64, 4) (8 rounds)
// 4.8 against 21, of (4096, 512, 4) 17 against 28, but of (2048, 512, 4) (4
// rounds) 16.9 against 15.3. In rows of under 4 outputs each of such a thread's
// loads fetches a cache line, so LDS pays sooner: (4096, 512, 2) 58 against 30
// us. Sums, argmax and argmin of more than COLS_MAX_ROUNDS go to threads at any
// length (a block's fold then takes longer than they do: argmax of (8192,
// 4096, 2) 447 against 826 us, its sum 446 against 518, its maxima 446 against 293).
constexpr int64_t COLS_ROUND_LEN = 128;
constexpr int64_t COLS_ROUND_LEN_NARROW = 64;
constexpr int64_t COLS_MAX_ROUNDS = 8;

// Other strided strips take a thread per output, its 16 loads in flight, or from
// VEC_MIN_OUT outputs a CU on, where a quarter of the threads still fill the
// chip, a thread per four, 8 float4s in flight: sums of (29, 75576) 5.2 us
// against 7.2, of (1000, 20480) 29.5 against 73.5, of (128, 327680) 25 against
// 29, but of (16, 655360) 8.5 against 7.4, of (4, 16777216) 92 against 55.
constexpr int64_t VEC_MIN_OUT = 2048;

constexpr bool is_arg(int k) { return k == OXI_REDUCE_ARGMAX || k == OXI_REDUCE_ARGMIN; }
// kinds whose result depends on the order of the fold
constexpr bool is_fold(int k) { return k == OXI_REDUCE_SUM || k == OXI_REDUCE_MEAN || k == OXI_REDUCE_NORM; }

// Drops dims of size 1 and merges dims that lie one after the other in memory:
// the outputs stay in their row-major order, and the rules below see how many
// of them are adjacent.
inline void simplify(RPlan& p) {
  int nd = 0;
  for (int d = 0; d < p.nd; ++d) {
    if (p.size[d] == 1) continue;
    if (nd && p.st[nd - 1] == p.st[d] * p.size[d]) {
      p.size[nd - 1] *= p.size[d];
      p.st[nd - 1] = p.st[d];
    } else {
      p.size[nd] = p.size[d];
      p.st[nd] = p.st[d];
      ++nd;
    }
  }
  p.nd = nd;
}

enum class ReduceKernel { Parts, Strips, Cols, Vec, Threads };

struct ReduceRoute {
  ReduceKernel kernel;
  int threads;            // of a block (Strips: of a strip; 64: four strips to a block of 256)
  int64_t blocks;
  int64_t part, parts;    // Parts: positions in a part, parts in a strip
  int64_t inner, groups;  // Cols: adjacent outputs in a row, blocks in a row
  bool vec;               // Cols: float4 rows
};

// The launch of a simplified plan.
inline ReduceRoute reduce_route(int kind, const RPlan& p, int64_t nout, const float* x, const float* out, int cus) {
  const auto ceil = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const auto aligned = [](const float* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
  ReduceRoute r{};
  if (p.rst == 1 && p.len >= 32) {
    if (nout < cus && p.len >= SPLIT_MIN_LEN) {
      const int64_t want = std::min(ceil(SPLIT_BLOCKS_PER_CU * (int64_t)cus, nout), SPLIT_MAX_PARTS);
      r.kernel = ReduceKernel::Parts;
      r.threads = 256;
      r.part = ceil(ceil(p.len, want), SPLIT_MIN_PART) * SPLIT_MIN_PART;
      r.parts = ceil(p.len, r.part);
      r.blocks = nout * r.parts;
      return r;
    }
    r.kernel = ReduceKernel::Strips;
    r.threads = p.len <= WAVE_MAX_LEN || !grid_fits(nout, 256) ? 64 : nout < 2 * cus ? 1024 : 256;
    r.blocks = r.threads == 64 ? ceil(nout, 256 / 64) : nout;
    if (grid_fits(r.blocks, std::max(r.threads, 256))) return r;
  }
  const bool unit = p.nd > 0 && p.st[p.nd - 1] == 1;  // outputs adjacent in memory
  r.inner = unit ? p.size[p.nd - 1] : 1;
  // rows of float4s: every row start 16-byte aligned
  r.vec = unit && r.inner % 4 == 0 && p.rst % 4 == 0 && aligned(x);
  for (int d = 0; d + 1 < p.nd && r.vec; ++d)
    if (p.st[d] % 4) r.vec = false;
  r.threads = 256;
  if (p.len >= COLS_MIN_LEN && nout <= COLS_MAX_OUT) {
    r.groups = ceil(r.inner, COLS_C);
    r.blocks = nout / r.inner * r.groups;
    const int64_t round = 2 * (int64_t)cus;
    const int64_t per_round = r.inner < 4 ? COLS_ROUND_LEN_NARROW : COLS_ROUND_LEN;
    const int64_t most = is_fold(kind) || is_arg(kind) ? COLS_MAX_ROUNDS * round : COLS_MAX_OUT;
    if (r.blocks <= round || (r.blocks <= most && p.len * round >= per_round * r.blocks)) {
      r.kernel = ReduceKernel::Cols;
      r.threads = COLS_THREADS;
      return r;
    }
  }
  r.kernel = !is_arg(kind) && r.vec && aligned(out) && nout >= VEC_MIN_OUT * (int64_t)cus ? ReduceKernel::Vec
                                                                                         : ReduceKernel::Threads;
  r.blocks = std::min(ceil(r.kernel == ReduceKernel::Vec ? nout / 4 : nout, 256), (int64_t)cus * 64);
  return r;
}

}  // namespace oxi
