// Softmax, log-softmax and fused cross-entropy kernels for gfx950.
//
// Softmax-family ops reduce over the middle dim of a contiguous
// (outer, len, inner) buffer. inner == 1 (the last dim, the hot case) runs one
// row per row group with the row held in registers when it fits
// (len <= 8192, 16-byte aligned), so x is read once and y written once;
// longer rows stream twice (online max/sum pass, then the write pass).
// inner > 1 runs tiles of adjacent columns, their positions spread over the
// block and held in registers.
//
// Cross-entropy (mean reduction) is fused into two kernels: the forward streams
// each logits row once with an online (max, sum-exp) and writes the row's
// log-sum-exp plus its picked log-probability; a one-block kernel forms the
// mean in float64 in fixed order. The backward streams logits once more and
// writes (softmax - onehot) * g / n. Bytes per row: 1 read fwd, 1 read + 1
// write bwd, instead of the reference's dense one-hot and ~16 passes
// (python/oxitorch/nn/functional.py:277-293).
#include <algorithm>
#include <cmath>

#include "internal.h"
#include "rowtile.h"
#include "softmax_mid.h"

namespace oxi {
namespace {

constexpr int BS = 256;

// Running (max, sum of exp(v - max)) of one thread; `m == -inf` means no
// finite contribution yet (sum 0).
struct Online {
  float m = NEG_INF;
  float s = 0.f;
  __device__ __forceinline__ void add4(const f4& v) {
    const float cm = max4(v);
    if (cm > m) {
      s = (m == NEG_INF) ? 0.f : s * expf(m - cm);
      m = cm;
    }
    if (m != NEG_INF) s += sum4(exp4(v - m));
    else if (cm != cm || v.x != v.x || v.y != v.y || v.z != v.z || v.w != v.w) s = __builtin_nanf("");
  }
  __device__ __forceinline__ void add1(float v) {
    if (v > m) {
      s = (m == NEG_INF) ? 0.f : s * expf(m - v);
      m = v;
    }
    if (m != NEG_INF) s += expf(v - m);
    else if (v != v) s = __builtin_nanf("");
  }
};

// Combine the Online states of a row group; every thread gets (M, S).
template <int TPR>
__device__ __forceinline__ void group_online(Online& o, float* lds) {
  const float M = group_max<TPR>(o.m, lds);
  float part = (o.m == NEG_INF) ? ((o.s != o.s) ? o.s : 0.f) : o.s * expf(o.m - M);
  const float S = group_sum<TPR, float>(part, lds + TPR / 64);
  o.m = M;
  o.s = S;
}

// ---------------------------------------------------------------------------
// Last-dim kernels, register-resident rows.

template <int TPR, int NV, bool LOG, bool NTS, bool FULL>
__global__ __launch_bounds__((row_block_threads(TPR))) void sm_fwd_k(const float* __restrict__ x, float* __restrict__ y,
                                                                  int64_t rows, int H_arg) {
  const int H = FULL ? 4 * TPR * NV : H_arg;  // FULL: rows of exactly TPR * NV float4s
  constexpr int NT = row_block_threads(TPR);
  constexpr int GPB = NT / TPR;
  __shared__ float lds[2 * (NT / 64)];
  const int t = threadIdx.x % TPR;
  const int64_t row = (int64_t)blockIdx.x * GPB + threadIdx.x / TPR;
  if (row >= rows) return;
  const int h4 = H >> 2;
  RowTile<TPR, NV> xt;
  xt.load(x + row * H, h4, t);
  float m = NEG_INF;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if (k * TPR + t < h4) m = fmaxf(m, max4(xt.v[k]));
  m = group_max_once<TPR>(m, lds);  // one row per block: one barrier per reduction
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    if (k * TPR + t < h4) {
      const f4 z = xt.v[k] - m;
      const f4 e = exp4(z);
      s += sum4(e);
      xt.v[k] = LOG ? z : e;
    }
  }
  s = group_sum_once<TPR, float>(s, lds + NT / 64);
  if constexpr (LOG) {
    const float L = logf(s);
#pragma unroll
    for (int k = 0; k < NV; ++k) xt.v[k] = xt.v[k] - L;
  } else {
    div_by_sum<NV>(xt.v, s);  // e / s, rounded as the division operator rounds it
  }
  xt.template store<NTS>(y + row * H, h4, t);
}

template <int TPR, int NV, bool LOG, bool NTS, bool FULL>
__global__ __launch_bounds__((row_block_threads(TPR))) void sm_bwd_k(const float* __restrict__ y, const float* __restrict__ g,
                                                                  float* __restrict__ dx, int64_t rows, int H_arg) {
  const int H = FULL ? 4 * TPR * NV : H_arg;  // FULL: rows of exactly TPR * NV float4s
  constexpr int NT = row_block_threads(TPR);
  constexpr int GPB = NT / TPR;
  __shared__ float lds[NT / 64];
  const int t = threadIdx.x % TPR;
  const int64_t row = (int64_t)blockIdx.x * GPB + threadIdx.x / TPR;
  if (row >= rows) return;
  const int h4 = H >> 2;
  RowTile<TPR, NV> yt, gt;
  yt.load(y + row * H, h4, t);
  gt.load(g + row * H, h4, t);
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) s += LOG ? sum4(gt.v[k]) : sum4(gt.v[k] * yt.v[k]);
  s = group_sum_once<TPR, float>(s, lds);  // the block's only reduction
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    if constexpr (LOG) gt.v[k] = gt.v[k] - exp4(yt.v[k]) * s;
    else gt.v[k] = yt.v[k] * (gt.v[k] - s);
  }
  gt.template store<NTS>(dx + row * H, h4, t);
}

// Last-dim kernels for any length / alignment: one block per row, two passes.
template <bool LOG>
__global__ __launch_bounds__(BS) void sm_fwd_loop_k(const float* __restrict__ x, float* __restrict__ y, int64_t rows, int H) {
  __shared__ float lds[2 * (BS / 64)];
  const int64_t row = blockIdx.x;
  const float* xr = x + row * H;
  Online o;
  for (int c = threadIdx.x; c < H; c += BS) o.add1(xr[c]);
  group_online<BS>(o, lds);
  float* yr = y + row * H;
  const float L = logf(o.s);
  for (int c = threadIdx.x; c < H; c += BS) {
    const float z = xr[c] - o.m;
    yr[c] = LOG ? z - L : expf(z) / o.s;
  }
}

template <bool LOG>
__global__ __launch_bounds__(BS) void sm_bwd_loop_k(const float* __restrict__ y, const float* __restrict__ g,
                                                    float* __restrict__ dx, int64_t rows, int H) {
  __shared__ float lds[BS / 64];
  const int64_t row = blockIdx.x;
  const float* yr = y + row * H;
  const float* gr = g + row * H;
  float s = 0.f;
  for (int c = threadIdx.x; c < H; c += BS) s += LOG ? gr[c] : gr[c] * yr[c];
  s = group_sum<BS, float>(s, lds);
  float* d = dx + row * H;
  for (int c = threadIdx.x; c < H; c += BS) d[c] = LOG ? gr[c] - expf(yr[c]) * s : yr[c] * (gr[c] - s);
}

// ---------------------------------------------------------------------------
// Middle-dim kernels (inner > 1). A block owns TX units of W adjacent columns
// (4, or single columns when inner < 4) and spreads their len positions over
// TY threads a unit, NV positions a thread: up to TY * NV positions are held
// in registers, so x crosses HBM once and the columns' maxima and sums are
// combined through LDS; longer columns (NV = 0) are streamed twice, MID_U
// positions in flight a thread, with an online maximum and sum. What bounds
// the first is a block's one round of loads, compute and stores with little
// else on its CU meanwhile: with the inputs in HBM the log-softmax of (16, 150,
// 4096) takes 23.4 us forward (3.4 TB/s) and 25.1 us backward (4.7). A row's last unit starts at inner - W, so it may repeat columns of the
// one before: both form and write the same values. TX and TY are chosen on the
// host (mid_shape): wide tiles for few positions, 128 bytes of a row (TX = 8)
// for many. Against one thread a column walking it twice, the same with its
// inputs in the Infinity Cache takes 14.6 us forward and 20.4 us backward
// instead of 115 and 92, of (2, 2846, 1901), streamed, 73 and 59 instead of
// 1800 and 1500, of (65536, 8, 3) 7.7 and 8.4 instead of 8.9 and 9.8. Plain
// loads: a row's 128-byte lines are shared by tiles when inner is odd, and
// non-temporal ones took 21 and 27 us at (16, 150, 4096) with the input in the
// Infinity Cache (from HBM: 45.6 us for both against 48.0). 12 positions a
// thread instead of 8: 15.7 against 21.2 us there with those loads, and slower
// below 64 positions.

constexpr int MID_U = 4;

template <int W>
struct Lanes {  // W columns' values
  typedef float type __attribute__((ext_vector_type(W), aligned(4)));
};
template <>
struct Lanes<1> {
  typedef float type;
};

// The unit of this thread.
struct MidUnit {
  int tx, ty;     // its place in the block's tile
  bool act;       // it has positions of an existing unit
  int64_t base;   // its first column's position 0
};

// Unit id: the units of every outer index, one after another.
template <int W>
__device__ __forceinline__ MidUnit mid_unit(int64_t len, int64_t inner, int64_t units, int64_t total, int TX) {
  MidUnit m;
  m.tx = threadIdx.x % TX;
  m.ty = threadIdx.x / TX;
  const int64_t id = (int64_t)blockIdx.x * TX + m.tx;
  m.act = id < total;
  const int64_t o = id / units, u = id % units;
  m.base = o * len * inner + min<int64_t>(u * W, inner - W);
  return m;
}

// op over the TY threads of every unit; each gets the result. `red` holds a
// value per thread and is free again after the call.
template <class V, class Op>
__device__ __forceinline__ V mid_combine(V v, V* red, const MidUnit& m, int TX, int TY, Op op) {
  if (TY == 1) return v;
  red[m.ty * TX + m.tx] = v;
  for (int h = TY >> 1; h >= 1; h >>= 1) {  // TY is a power of two
    __syncthreads();
    if (m.ty < h) red[m.ty * TX + m.tx] = op(red[m.ty * TX + m.tx], red[(m.ty + h) * TX + m.tx]);
  }
  __syncthreads();
  v = red[m.tx];
  __syncthreads();
  return v;
}

template <int W>
__device__ __forceinline__ float& at(typename Lanes<W>::type& v, int j) {
  return reinterpret_cast<float*>(&v)[j];
}

template <bool LOG, int W, int NV, int NT>
__global__ __launch_bounds__(NT) void sm_fwd_mid_k(const float* __restrict__ x, float* __restrict__ y, int64_t len,
                                                   int64_t inner, int64_t units, int64_t total, int TX, int TY) {
  using V = typename Lanes<W>::type;
  constexpr int N = NV ? NV : MID_U;
  __shared__ V red[NT];
  const MidUnit u = mid_unit<W>(len, inner, units, total, TX);
  const float* xc = x + u.base;
  float* yc = y + u.base;
  auto each = [](auto f) {
#pragma unroll
    for (int j = 0; j < W; ++j) f(j);
  };
  auto vmax = [&](V a, V b) {
    each([&](int j) { at<W>(a, j) = fmaxf(at<W>(a, j), at<W>(b, j)); });
    return a;
  };
  auto vsum = [](V a, V b) { return a + b; };
  V v[N];
  // positions k0 + ty, + TY, ...: those past the end give -inf, which counts for nothing
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int64_t k = k0 + u.ty + (int64_t)i * TY;
      each([&](int j) { at<W>(v[i], j) = NEG_INF; });
      if (u.act && k < len) v[i] = *reinterpret_cast<const V*>(xc + k * inner);
    }
  };
  V m, s;
  each([&](int j) {
    at<W>(m, j) = NEG_INF;
    at<W>(s, j) = 0.f;
  });
  if constexpr (NV > 0) {
    load(0);
#pragma unroll
    for (int i = 0; i < N; ++i) m = vmax(m, v[i]);
  } else {
    for (int64_t k0 = 0; k0 < len; k0 += (int64_t)N * TY) {
      load(k0);
      each([&](int j) {
        float cm = at<W>(m, j);
#pragma unroll
        for (int i = 0; i < N; ++i) cm = fmaxf(cm, at<W>(v[i], j));
        const float ref = cm == NEG_INF ? 0.f : cm;
        float acc = at<W>(s, j) * exp_le0(at<W>(m, j) - ref);
#pragma unroll
        for (int i = 0; i < N; ++i) acc += exp_le0(at<W>(v[i], j) - ref);
        at<W>(s, j) = acc;
        at<W>(m, j) = cm;
      });
    }
  }
  const V M = mid_combine(m, red, u, TX, TY, vmax);
  if constexpr (NV > 0) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (u.ty + (int64_t)i * TY < len)
        each([&](int j) {
          V Mv = M;
          const float z = at<W>(v[i], j) - at<W>(Mv, j);
          const float e = exp_le0(z);
          at<W>(s, j) += e;
          at<W>(v[i], j) = LOG ? z : e;
        });
  } else {
    each([&](int j) {
      V Mv = M;
      const float ref = at<W>(Mv, j) == NEG_INF ? 0.f : at<W>(Mv, j);
      at<W>(s, j) *= exp_le0(at<W>(m, j) - ref);
    });
  }
  V S = mid_combine(s, red, u, TX, TY, vsum);
  V out;
  auto finish = [&](V e) {  // from z or e (NV > 0), or from x
    V Mv = M;
    each([&](int j) {
      if constexpr (NV == 0) {
        const float z = at<W>(e, j) - at<W>(Mv, j);
        at<W>(out, j) = LOG ? z - logf(at<W>(S, j)) : exp_le0(z) / at<W>(S, j);
      } else {
        at<W>(out, j) = LOG ? at<W>(e, j) - at<W>(S, j) : at<W>(e, j) / at<W>(S, j);
      }
    });
    return out;
  };
  if (!u.act) return;
  if constexpr (NV > 0) {
    if constexpr (LOG) each([&](int j) { at<W>(S, j) = logf(at<W>(S, j)); });
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int64_t k = u.ty + (int64_t)i * TY;
      if (k < len) *reinterpret_cast<V*>(yc + k * inner) = finish(v[i]);
    }
  } else {
    for (int64_t k0 = u.ty; k0 < len; k0 += (int64_t)N * TY) {
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (k0 + (int64_t)i * TY < len) v[i] = *reinterpret_cast<const V*>(xc + (k0 + (int64_t)i * TY) * inner);
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (k0 + (int64_t)i * TY < len) *reinterpret_cast<V*>(yc + (k0 + (int64_t)i * TY) * inner) = finish(v[i]);
    }
  }
}

template <bool LOG, int W, int NV, int NT>
__global__ __launch_bounds__(NT) void sm_bwd_mid_k(const float* __restrict__ y, const float* __restrict__ g,
                                                   float* __restrict__ dx, int64_t len, int64_t inner, int64_t units,
                                                   int64_t total, int TX, int TY) {
  using V = typename Lanes<W>::type;
  constexpr int N = NV ? NV : MID_U;
  __shared__ V red[NT];
  const MidUnit u = mid_unit<W>(len, inner, units, total, TX);
  const float *yc = y + u.base, *gc = g + u.base;
  float* dc = dx + u.base;
  V a[N], b[N];  // y and g; 0 past the end
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int64_t k = k0 + u.ty + (int64_t)i * TY;
      a[i] = V{};
      b[i] = V{};
      if (u.act && k < len) {
        a[i] = *reinterpret_cast<const V*>(yc + k * inner);
        b[i] = *reinterpret_cast<const V*>(gc + k * inner);
      }
    }
  };
  V s = V{};
  for (int64_t k0 = 0; k0 < len; k0 += (int64_t)N * TY) {
    load(k0);
#pragma unroll
    for (int i = 0; i < N; ++i) s = s + (LOG ? b[i] : b[i] * a[i]);
    if constexpr (NV > 0) break;
  }
  const V S = mid_combine(s, red, u, TX, TY, [](V p, V q) { return p + q; });
  if (!u.act) return;
  for (int64_t k0 = 0; k0 < len; k0 += (int64_t)N * TY) {
    if constexpr (NV == 0) load(k0);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int64_t k = k0 + u.ty + (int64_t)i * TY;
      if (k >= len) continue;
      V o;
      if constexpr (LOG) {
#pragma unroll
        for (int j = 0; j < W; ++j) at<W>(o, j) = exp_le0(at<W>(a[i], j));
        o = b[i] - o * S;
      } else {
        o = a[i] * (b[i] - S);
      }
      *reinterpret_cast<V*>(dc + k * inner) = o;
    }
    if constexpr (NV > 0) break;
  }
}

// ---------------------------------------------------------------------------
// Cross-entropy.

constexpr int CE_BS = 256;
constexpr int CE_U = 4;   // forward: float4 loads in flight per thread per step
constexpr int CE_SHORT = 320;  // forward: odd rows of up to this many classes go a float a thread
constexpr int CE_BU = 1;  // backward: float4s per thread (one per thread streams fastest)

// The reference picks the target's log-probability as
// sum(onehot * log_softmax(x)) (functional.py:287-292): a non-target class
// whose log-probability is -inf (x - max == -inf: a -inf logit, or one so far
// below the max that the difference overflows) contributes 0 * -inf = NaN,
// so that row's picked value, and the loss, is NaN. `mn` is the row's
// minimum over its non-target logits; x - max is monotone in x.
__device__ __forceinline__ bool onehot_nan(float mn, float m) { return mn - m == NEG_INF; }

// v with component j replaced by +inf (out of a minimum).
__device__ __forceinline__ f4 drop_lane(const f4& v, int j) {
  const float P = -NEG_INF;
  return f4{j == 0 ? P : v.x, j == 1 ? P : v.y, j == 2 ? P : v.z, j == 3 ? P : v.w};
}

// Rows the register-row kernel does not take (more than 16384 float4s, or not
// a multiple of 4 classes at a 16-byte address): one block per row, streaming
// it with CE_U float4s in flight a thread, at whatever float alignment the row
// has, and the last C % 4 logits on their own. HBM bounds it: 4096 rows of
// 50257 classes take 136-160 us (5.1-6.0 TB/s) where single floats took 330.
// SHORT: rows of up to CE_SHORT classes, a float a thread: most threads have
// no float4 of theirs, and the others' chains and the tail are what the block
// waits for (rows of 33 classes at (127100, 33) 137 us against 171 as float4s,
// of 301 at (55738, 301) 77 against 80; of 385 at (43577, 385) 63.5 against 62.6).
// lse[row] = max + log(sum exp(x - max));
// picked[row] = (x[t] - max) - log(sum)  (the reference's ls[row, t]), or
// NaN where the reference's one-hot product makes it NaN (onehot_nan).
template <int NT, bool SHORT>
__global__ __launch_bounds__(NT) void ce_fwd_k(const float* __restrict__ logits, const int64_t* __restrict__ targets,
                                               float* __restrict__ lse, float* __restrict__ picked, int64_t n, int C,
                                               int* __restrict__ guard) {
  __shared__ float lds[2 * (NT / 64)];
  const int64_t row = blockIdx.x;
  const float* xr = logits + row * C;
  int64_t tg = targets[row];
  const bool bad = tg < 0 || tg >= C;
  if (bad) tg = 0;
  float mn = -NEG_INF;
  Online o;
  if constexpr (SHORT) {
    for (int c = threadIdx.x; c < C; c += NT) {
      const float v = xr[c];
      o.add1(v);
      if (c != tg) mn = fminf(mn, v);
    }
  } else {
    const f4u* p = reinterpret_cast<const f4u*>(xr);
    const int c4 = C >> 2;
    const int ct = (int)(tg >> 2);
    const int jt = (int)(tg & 3);
    int c = threadIdx.x;
    for (; c + (CE_U - 1) * NT < c4; c += CE_U * NT) {
      f4 v[CE_U];
#pragma unroll
      for (int u = 0; u < CE_U; ++u) v[u] = ld_stream(p + c + u * NT);
#pragma unroll
      for (int u = 0; u < CE_U; ++u) mn = fminf(mn, min4(c + u * NT == ct ? drop_lane(v[u], jt) : v[u]));
      float cm = max4(v[0]);
#pragma unroll
      for (int u = 1; u < CE_U; ++u) cm = fmaxf(cm, max4(v[u]));
      if (cm > o.m) {
        o.s = (o.m == NEG_INF) ? 0.f : o.s * expf(o.m - cm);
        o.m = cm;
      }
      if (o.m != NEG_INF) {
        float acc = 0.f;
#pragma unroll
        for (int u = 0; u < CE_U; ++u) acc += sum4(exp4(v[u] - o.m));
        o.s += acc;
      } else {
#pragma unroll
        for (int u = 0; u < CE_U; ++u) o.add4(v[u]);
      }
    }
    for (; c < c4; c += NT) {
      const f4 v = p[c];
      o.add4(v);
      mn = fminf(mn, min4(c == ct ? drop_lane(v, jt) : v));
    }
    if ((int)threadIdx.x < (C & 3)) {
      const int e = 4 * c4 + threadIdx.x;
      const float v = xr[e];
      o.add1(v);
      if (e != tg) mn = fminf(mn, v);
    }
  }
  group_online<NT>(o, lds);
  mn = -group_max<NT>(-mn, lds);
  if (threadIdx.x == 0) {
    if (bad) atomicOr(guard, 1);
    const float L = logf(o.s);
    lse[row] = o.m + L;
    picked[row] = onehot_nan(mn, o.m) ? __builtin_nanf("") : (xr[tg] - o.m) - L;
  }
}

// Rows of up to RT * NV float4s, a row per block held in registers, so each
// row crosses HBM once: the row max (with the non-target minimum that
// onehot_nan needs, in the same reduction) and the sum of e = exp(x - max)
// (two block reductions), lse and picked. With `dunit` set the block also writes, from
// the e it kept in the same registers, the gradient of the mean loss for an
// upstream gradient of exactly 1, as the composed log_softmax VJP forms it
// (functional.py:277-293 through ops.rs's exp/sum/log/sub VJPs):
// gS * e with gS = (1 / n) * (1 / s), and gS * e - 1 / n at the target, so a
// backward seeded with 1 has nothing left to compute. One exp per element:
// with a second exp(x - lse) for the gradient the kernel spent about 39 VALU
// instructions per element and ran at the VALU bound, not the HBM bound.
// The zero-sum residue the reference routes to the argmax (the max VJP) is
// rounding noise of the reference's own evaluation and is not formed.
// Measured at C3 (8192 x 32000), two-exp form: 512 x 16 ran the forward with
// the gradient in 380 us (1024 x 8, held to one block per CU by its 68 VGPRs:
// 476 us; 256 x 32: 417 us) and the forward alone in 181 us (streaming: 174 us).
// With one exp, the restructured loops below and 60 VGPRs, 1024 x 8 runs two
// blocks per CU and is the faster shape at C3 (see ce_forward).
// TAIL1: the row fills all but the last of a thread's NV float4 slots
// ((NV - 1) * RT < C / 4 <= NV * RT, as at C3's 32000 classes), so only slot
// NV - 1 is bounds-checked. The hot loops take the minimum over every logit;
// the reference's NaN rule needs the minimum over the non-target ones, which
// is formed again, with the target dropped, only for a row whose minimum
// could make it NaN. The target's logit comes from the owning thread's
// registers.
template <int RT, int NV, bool GRAD, bool NTS, bool TAIL1>
__global__ __launch_bounds__(RT) void ce_fwd_rows_k(const float* __restrict__ logits,
                                                    const int64_t* __restrict__ targets, float* __restrict__ lse,
                                                    float* __restrict__ picked, float* __restrict__ dunit, int64_t n,
                                                    int C, int* __restrict__ guard) {
  // slot sets: the max and the minimum, then the sum, then the rare
  // non-target minimum
  __shared__ float lds[4 * (RT / 64)];
  __shared__ float tlogit;
  const int64_t row = blockIdx.x;
  const int t = threadIdx.x;
  const int c4 = C >> 2;
  const float* xr = logits + row * C;
  const f4* p = reinterpret_cast<const f4*>(xr);
  auto in_row = [&](int k) { return (TAIL1 && k < NV - 1) || k * RT + t < c4; };
  f4 v[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * RT + t;
    v[k] = in_row(k) ? ld_stream(p + c) : f4{NEG_INF, NEG_INF, NEG_INF, NEG_INF};
  }
  int64_t tg = targets[row];
  const bool bad = tg < 0 || tg >= C;
  if (bad) tg = 0;
  // The target's float4 is slot kt of lane `own`; component jt.
  const int ct = (int)(tg >> 2);
  const int kt = ct / RT;
  const bool own = ct - kt * RT == t;
  const int jt = (int)(tg & 3);
  float m = NEG_INF;
  float mn = -NEG_INF;  // minimum over the row's logits (padding lanes hold -inf: skipped)
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    m = fmaxf(m, max4(v[k]));
    if (in_row(k)) mn = fminf(mn, min4(v[k]));
    if (k == kt) {
      if (own) tlogit = jt == 0 ? v[k].x : jt == 1 ? v[k].y : jt == 2 ? v[k].z : v[k].w;
    }
  }
  float nmn = -mn;
  group_max2_once<RT>(m, nmn, lds);
  const float ms = m == NEG_INF ? 0.f : m;
  // the row can be NaN only if its minimum is: then the minimum without the
  // target decides (block-uniform branch)
  bool nan_row = onehot_nan(-nmn, m);
  if (nan_row) {
    float mt = -NEG_INF;
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (in_row(k)) mt = fminf(mt, min4(k == kt && own ? drop_lane(v[k], jt) : v[k]));
    float nmt = -mt;
    nmt = group_max_once<RT>(nmt, lds + 3 * (RT / 64));
    nan_row = onehot_nan(-nmt, m);
  }
  // Lanes past the row hold -inf: their e is exp(-inf) = 0 and adds nothing.
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    v[k] = exp4(v[k] - ms);
    s += sum4(v[k]);
  }
  s = group_sum_once<RT, float>(s, lds + 2 * (RT / 64));  // its barrier also publishes tlogit
  if constexpr (RT == 64) __syncthreads();                 // (one wave: no barrier in the reduction)
  const float L = logf(s);
  if (t == 0) {
    if (bad) atomicOr(guard, 1);
    lse[row] = m + L;
    picked[row] = nan_row ? __builtin_nanf("") : (tlogit - m) - L;
  }
  if constexpr (GRAD) {
    const float scale = 1.0f / (float)n;
    const float gs = scale * (1.0f / s);
    f4* q = reinterpret_cast<f4*>(dunit + row * C);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = k * RT + t;
      if (in_row(k)) {
        f4 d = v[k] * gs;
        if (k == kt) {
          if (own) {
            if (jt == 0) d.x -= scale;
            else if (jt == 1) d.y -= scale;
            else if (jt == 2) d.z -= scale;
            else d.w -= scale;
          }
        }
        st_stream<NTS>(d, q + c);
      }
    }
  }
}

// loss[0] = -(sum(picked) / n), sum in float64 in fixed order.
__global__ __launch_bounds__(1024) void ce_mean_k(const float* __restrict__ picked, int64_t n, float* __restrict__ loss) {
  __shared__ double s[1024];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) acc += (double)picked[i];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 512; w >= 1; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = -((float)s[0] / (float)n);
}

// dlogits = (exp(x - lse) - onehot) * (g / n). Grid: (column blocks, rows).
template <bool NTS>
__global__ __launch_bounds__(CE_BS) void ce_bwd_k(const float* __restrict__ logits, const int64_t* __restrict__ targets,
                                                  const float* __restrict__ lse, const float* __restrict__ gloss,
                                                  float* __restrict__ dlogits, int64_t n, int C, int vec) {
  const int64_t row = blockIdx.y;
  const float scale = gloss[0] / (float)n;
  const float l = lse[row];
  int64_t t = targets[row];
  const float* xr = logits + row * C;
  float* dr = dlogits + row * C;
  if (vec) {
    const f4* p = reinterpret_cast<const f4*>(xr);
    f4* q = reinterpret_cast<f4*>(dr);
    const int c4 = C >> 2;
    const int per_block = CE_BS * CE_BU;
    const int c0 = blockIdx.x * per_block + threadIdx.x;
    f4 v[CE_BU];
#pragma unroll
    for (int u = 0; u < CE_BU; ++u) {
      const int c = c0 + u * CE_BS;
      if (c < c4) v[u] = ld_stream(p + c);
    }
#pragma unroll
    for (int u = 0; u < CE_BU; ++u) {
      const int c = c0 + u * CE_BS;
      if (c < c4) {
        f4 e = exp4(v[u] - l);
        const int64_t base = (int64_t)c * 4;
        if (t >= base && t < base + 4) {
          const int j = (int)(t - base);
          if (j == 0) e.x -= 1.f;
          else if (j == 1) e.y -= 1.f;
          else if (j == 2) e.z -= 1.f;
          else e.w -= 1.f;
        }
        st_stream<NTS>(e * scale, q + c);
      }
    }
  } else if (C <= CE_BS) {
    // short odd rows: a float a thread, in one block (a float4 a thread leaves
    // three quarters of it idle: (127100, 33) 59 us against 67, (65793, 255) 34
    // against 45, but (65280, 257), two blocks a row, 58 against 42)
    const int c = threadIdx.x;
    if (c < C) {
      float e = exp_le0(xr[c] - l);
      if (c == t) e -= 1.f;
      dr[c] = e * scale;
    }
  } else {
    // Rows at any float alignment: the gradient's 16-byte granules, whole in
    // the row, are a float4 each (the logits' share their phase unless the
    // buffers differ in it); the up to 3 classes before the first and after
    // the last go one each to the first block's threads. (4096, 50257) takes
    // 264-275 us (6.0-6.2 TB/s) where a float a thread took 550.
    const int head = min((int)((0 - (reinterpret_cast<uintptr_t>(dr) >> 2)) & 3u), C);
    const int c4 = (C - head) >> 2;
    static_assert(CE_BU == 1, "odd rows: one float4 a thread, as the grid has them");
    const int c = blockIdx.x * CE_BS + threadIdx.x;
    if (c < c4) {
      const int e0 = head + 4 * c;
      f4 e = exp4(ld_stream(reinterpret_cast<const f4u*>(xr + e0)) - l);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (e0 + j == t) e[j] -= 1.f;
      st_stream<NTS>(e * scale, reinterpret_cast<f4*>(dr + e0));
    }
    if (blockIdx.x == 0 && threadIdx.x < 6) {
      const int k = threadIdx.x;
      const int e0 = k < 3 ? k : head + 4 * c4 + (k - 3);
      if (k < 3 ? e0 < head : e0 < C) {
        float e = exp_le0(xr[e0] - l);
        if (e0 == t) e -= 1.f;
        dr[e0] = e * scale;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Host dispatch.


bool aligned16(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if (reinterpret_cast<uintptr_t>(p) & 15u) return false;
  return true;
}

int check_olen(const char* what, int64_t outer, int64_t len, int64_t inner, std::initializer_list<const void*> ps) {
  if (outer < 0 || len < 0 || inner < 0)
    return fail(OXI_INVALID_ARGUMENT, "%s: negative size", what);
  // len and outer * inner each bounded, and the element count inside int64
  const int64_t lim = (int64_t)1 << 40;
  if (len > ((int64_t)1 << 30) || (outer && inner > lim / outer) ||
      (outer && inner && len > (((int64_t)1 << 60) / outer) / inner))
    return fail(OXI_INVALID_ARGUMENT, "%s: size exceeds the kernel limits", what);
  if (outer && len && inner)
    for (const void* p : ps)
      if (!p) return fail(OXI_INVALID_ARGUMENT, "%s: NULL tensor pointer", what);
  return OXI_OK;
}

#define OXI_MID_GO(K, W, NV, NT, ...)                                                                       \
  K<LOG, W, NV, NT><<<dim3((unsigned)m.blocks), dim3(NT), 0, s>>>(__VA_ARGS__, len, inner, m.units, m.total,   \
                                                                 m.tx, m.ty)
#define OXI_MID_W(K, W, FEW, MOST, ...)                                                                    \
  if (m.nv == 0) OXI_MID_GO(K, W, 0, 1024, __VA_ARGS__); /* mid_shape: streamed on 1024 threads only, */   \
  else if (m.nv == FEW) OXI_MID_GO(K, W, FEW, 256, __VA_ARGS__); /* few positions on 256 only */           \
  else if (m.nt == 256) OXI_MID_GO(K, W, MOST, 256, __VA_ARGS__);                                          \
  else OXI_MID_GO(K, W, MOST, 1024, __VA_ARGS__);
#define OXI_MID(K, ...)                                                                                    \
  if (inner >= 4) {                                                                                        \
    OXI_MID_W(K, 4, 2, 8, __VA_ARGS__)                                                                     \
  } else {                                                                                                 \
    OXI_MID_W(K, 1, 4, 16, __VA_ARGS__)                                                                    \
  }

template <bool LOG>
int launch_fwd(const float* x, float* y, int64_t outer, int64_t len, int64_t inner) {
  hipStream_t s = stream();
  if (inner == 1) {
    const int cfg = (len % 4 == 0 && aligned16({x, y})) ? pick_row_cfg(len / 4) : 0;
    const int h = (int)len;
    const bool nts = nt_stores(outer * len * 4);
#define OXI_SMF_GO(TPR, NV, NTS, FULL)                                                                  \
  sm_fwd_k<TPR, NV, LOG, NTS, FULL><<<dim3((unsigned)ceil_div(outer, row_block_threads(TPR) / TPR)),         \
                                     dim3(row_block_threads(TPR)), 0, s>>>(x, y, outer, h)
#define OXI_SMF(TPR, NV)                                                                                   \
  case TPR * 10 + NV:                                                                                      \
    if (h == 4 * TPR * NV) {                                                                               \
      if (nts) OXI_SMF_GO(TPR, NV, true, true);                                                            \
      else OXI_SMF_GO(TPR, NV, false, true);                                                               \
    } else {                                                                                               \
      if (nts) OXI_SMF_GO(TPR, NV, true, false);                                                           \
      else OXI_SMF_GO(TPR, NV, false, false);                                                              \
    }                                                                                                      \
    break;
    switch (cfg) {
      OXI_SMF(64, 1)
      OXI_SMF(64, 2)
      OXI_SMF(64, 3)
      OXI_SMF(64, 4)
      OXI_SMF(256, 2)
      OXI_SMF(256, 4)
      OXI_SMF(256, 8)
                default:
        sm_fwd_loop_k<LOG><<<dim3((unsigned)outer), dim3(BS), 0, s>>>(x, y, outer, h);
    }
#undef OXI_SMF
#undef OXI_SMF_GO
  } else {
    for (int64_t o0 = 0, oc = mid_outer_max(len, inner); o0 < outer; o0 += oc) {
      const MidShape m = mid_shape(std::min(oc, outer - o0), len, inner);
      const int64_t at = o0 * len * inner;
      OXI_MID(sm_fwd_mid_k, x + at, y + at)
    }
  }
  return check_launch(LOG ? "log_softmax_fwd" : "softmax_fwd");
}

template <bool LOG>
int launch_bwd(const float* y, const float* g, float* dx, int64_t outer, int64_t len, int64_t inner) {
  hipStream_t s = stream();
  if (inner == 1) {
    const int cfg = (len % 4 == 0 && aligned16({y, g, dx})) ? pick_row_cfg(len / 4) : 0;
    const int h = (int)len;
    const bool nts = nt_stores(outer * len * 4);
#define OXI_SMB_GO(TPR, NV, NTS, FULL)                                                                  \
  sm_bwd_k<TPR, NV, LOG, NTS, FULL><<<dim3((unsigned)ceil_div(outer, row_block_threads(TPR) / TPR)),         \
                                     dim3(row_block_threads(TPR)), 0, s>>>(y, g, dx, outer, h)
#define OXI_SMB(TPR, NV)                                                                                   \
  case TPR * 10 + NV:                                                                                      \
    if (h == 4 * TPR * NV) {                                                                               \
      if (nts) OXI_SMB_GO(TPR, NV, true, true);                                                            \
      else OXI_SMB_GO(TPR, NV, false, true);                                                               \
    } else {                                                                                               \
      if (nts) OXI_SMB_GO(TPR, NV, true, false);                                                           \
      else OXI_SMB_GO(TPR, NV, false, false);                                                              \
    }                                                                                                      \
    break;
    switch (cfg) {
      OXI_SMB(64, 1)
      OXI_SMB(64, 2)
      OXI_SMB(64, 3)
      OXI_SMB(64, 4)
      OXI_SMB(256, 2)
      OXI_SMB(256, 4)
      OXI_SMB(256, 8)
                default:
        sm_bwd_loop_k<LOG><<<dim3((unsigned)outer), dim3(BS), 0, s>>>(y, g, dx, outer, h);
    }
#undef OXI_SMB
#undef OXI_SMB_GO
  } else {
    for (int64_t o0 = 0, oc = mid_outer_max(len, inner); o0 < outer; o0 += oc) {
      const MidShape m = mid_shape(std::min(oc, outer - o0), len, inner);
      const int64_t at = o0 * len * inner;
      OXI_MID(sm_bwd_mid_k, y + at, g + at, dx + at)
    }
  }
  return check_launch(LOG ? "log_softmax_bwd" : "softmax_bwd");
}

}  // namespace
}  // namespace oxi

using namespace oxi;

extern "C" {

int oxi_softmax_fwd(const float* x, float* y, int64_t outer, int64_t len, int64_t inner) {
  if (int rc = check_olen("softmax_fwd", outer, len, inner, {x, y})) return rc;
  if (outer == 0 || inner == 0 || len == 0) return OXI_OK;
  OXI_CHECK_INIT();
  return launch_fwd<false>(x, y, outer, len, inner);
}

int oxi_softmax_bwd(const float* y, const float* g, float* dx, int64_t outer, int64_t len, int64_t inner) {
  if (int rc = check_olen("softmax_bwd", outer, len, inner, {y, g, dx})) return rc;
  if (outer == 0 || inner == 0 || len == 0) return OXI_OK;
  OXI_CHECK_INIT();
  return launch_bwd<false>(y, g, dx, outer, len, inner);
}

int oxi_log_softmax_fwd(const float* x, float* y, int64_t outer, int64_t len, int64_t inner) {
  if (int rc = check_olen("log_softmax_fwd", outer, len, inner, {x, y})) return rc;
  if (outer == 0 || inner == 0 || len == 0) return OXI_OK;
  OXI_CHECK_INIT();
  return launch_fwd<true>(x, y, outer, len, inner);
}

int oxi_log_softmax_bwd(const float* y, const float* g, float* dx, int64_t outer, int64_t len, int64_t inner) {
  if (int rc = check_olen("log_softmax_bwd", outer, len, inner, {y, g, dx})) return rc;
  if (outer == 0 || inner == 0 || len == 0) return OXI_OK;
  OXI_CHECK_INIT();
  return launch_bwd<true>(y, g, dx, outer, len, inner);
}

}  // extern "C"

namespace oxi {
namespace {

// Loss and lse; with `dunit`, also the gradient for an upstream 1 (rows of
// c % 4 == 0 with 16-byte aligned operands only: NOT_IMPLEMENTED otherwise,
// before anything is launched).
int ce_forward(const char* what, const float* logits, const int64_t* targets, float* loss, float* lse, float* dunit,
               int64_t n, int64_t c) {
  if (n < 0 || c < 0) return fail(OXI_INVALID_ARGUMENT, "%s: negative size", what);
  if (!loss) return fail(OXI_INVALID_ARGUMENT, "%s: loss must not be NULL", what);
  if (c > ((int64_t)1 << 30) || n > ((int64_t)1 << 31) - 1)
    return fail(OXI_INVALID_ARGUMENT, "%s: size exceeds the kernel limits", what);
  OXI_CHECK_INIT();
  // picked.mean() of no rows: reduce_all's Mean of an empty strip is 0
  // (bindings lib.rs:126-143, ops.rs:247-249), and the loss is its negation
  if (n == 0) return oxi_fill(loss, 1, -0.0f);
  if (c == 0) return fail(OXI_INVALID_ARGUMENT, "%s: zero classes", what);
  if (!logits || !targets || !lse) return fail(OXI_INVALID_ARGUMENT, "%s: NULL tensor pointer", what);
  const int vec = (c % 4 == 0 && aligned16({logits})) ? 1 : 0;
  const int64_t c4 = c / 4;
  // (threads, float4s a thread) of the register-row kernel: 16 float4s a
  // thread, as few threads as the row needs; rows of 4097 to 8192 float4s
  // take 1024 threads of 8 (60 VGPRs, two blocks per CU): C3's step 362.6
  // and 362.7 us against 367.3 and 367.9 at 512 x 16 on one box.
  int rt = 0, nv = 16;
  if (vec) {
    if (c4 > 4096 && c4 <= 8192) {
      rt = 1024;
      nv = 8;
    } else {
      for (int t = 64; t <= 1024 && !rt; t *= 2)
        if (c4 <= (int64_t)t * 16) rt = t;
    }
  }
  if (dunit && !(rt && aligned16({dunit})))
    return fail(OXI_NOT_IMPLEMENTED, "%s: rows of %lld classes do not take the one-pass kernel (c %% 4 != 0, more "
                "than 65536 classes or unaligned)", what, (long long)c);
  Workspace picked(sizeof(float) * (size_t)n);
  if (!picked.p) return fail_alloc("cross_entropy_fwd: workspace");
  const dim3 grid((unsigned)n);
  float* pk = picked.as<float>();
  const bool nt = nt_stores(n * c * 4);  // the gradient's stores
  switch (rt * 100 + nv) {
#define OXI_CE_GO(RT, NV, GRAD, NTS, TAIL1)                                                                \
  ce_fwd_rows_k<RT, NV, GRAD, NTS, TAIL1><<<grid, dim3(RT), 0, stream()>>>(logits, targets, lse, pk, dunit, n, \
                                                                          (int)c, guard_flag())
#define OXI_CE_ROWS(RT, NV)                                                                                 \
  case RT * 100 + NV:                                                                                       \
    if (c4 > (NV - 1) * RT) {                                                                               \
      if (!dunit) OXI_CE_GO(RT, NV, false, false, true);                                                    \
      else if (nt) OXI_CE_GO(RT, NV, true, true, true);                                                     \
      else OXI_CE_GO(RT, NV, true, false, true);                                                            \
    } else {                                                                                                \
      if (!dunit) OXI_CE_GO(RT, NV, false, false, false);                                                   \
      else if (nt) OXI_CE_GO(RT, NV, true, true, false);                                                    \
      else OXI_CE_GO(RT, NV, true, false, false);                                                           \
    }                                                                                                       \
    break;
    OXI_CE_ROWS(64, 16)
    OXI_CE_ROWS(128, 16)
    OXI_CE_ROWS(256, 16)
    OXI_CE_ROWS(1024, 8)
    OXI_CE_ROWS(1024, 16)
#undef OXI_CE_ROWS
#undef OXI_CE_GO
    default:
      // fewer rows than two a CU: 1024 threads to a long row
      if (c <= CE_SHORT)
        ce_fwd_k<CE_BS, true><<<grid, dim3(CE_BS), 0, stream()>>>(logits, targets, lse, pk, n, (int)c, guard_flag());
      else if (n < 2 * cu_count() && c > 16384)
        ce_fwd_k<1024, false><<<grid, dim3(1024), 0, stream()>>>(logits, targets, lse, pk, n, (int)c, guard_flag());
      else
        ce_fwd_k<CE_BS, false><<<grid, dim3(CE_BS), 0, stream()>>>(logits, targets, lse, pk, n, (int)c, guard_flag());
  }
  if (int rc = check_launch(what)) return rc;
  ce_mean_k<<<1, 1024, 0, stream()>>>(picked.as<float>(), n, loss);
  return check_launch("cross_entropy_mean");
}

}  // namespace
}  // namespace oxi

extern "C" {

int oxi_cross_entropy_fwd(const float* logits, const int64_t* targets, float* loss, float* lse, int64_t n, int64_t c) {
  return ce_forward("cross_entropy_fwd", logits, targets, loss, lse, nullptr, n, c);
}

int oxi_cross_entropy_fwd_grad(const float* logits, const int64_t* targets, float* loss, float* lse, float* dlogits,
                               int64_t n, int64_t c) {
  if (!dlogits && n > 0 && c > 0) return fail(OXI_INVALID_ARGUMENT, "cross_entropy_fwd_grad: NULL dlogits");
  return ce_forward("cross_entropy_fwd_grad", logits, targets, loss, lse, n > 0 && c > 0 ? dlogits : nullptr, n, c);
}

int oxi_cross_entropy_bwd(const float* logits, const int64_t* targets, const float* lse, const float* gloss,
                          float* dlogits, int64_t n, int64_t c) {
  if (n < 0 || c < 0) return fail(OXI_INVALID_ARGUMENT, "cross_entropy_bwd: negative size");
  if (c > ((int64_t)1 << 30) || n > 65535LL * 32768LL)
    return fail(OXI_INVALID_ARGUMENT, "cross_entropy_bwd: size exceeds the kernel limits");
  if (n == 0 || c == 0) return OXI_OK;
  if (!logits || !targets || !lse || !gloss || !dlogits)
    return fail(OXI_INVALID_ARGUMENT, "cross_entropy_bwd: NULL tensor pointer");
  OXI_CHECK_INIT();
  const int vec = (c % 4 == 0 && aligned16({logits, dlogits})) ? 1 : 0;
  const int64_t units = std::max<int64_t>(1, c / 4);  // at least one block a row
  const unsigned gx = (unsigned)ceil_div(units, CE_BS * CE_BU);
  const bool nts = nt_stores(n * c * 4);
  if (n > 65535) {
    // grid.y is limited; launch row slabs
    for (int64_t r0 = 0; r0 < n; r0 += 65535) {
      const int64_t nr = (n - r0) < 65535 ? (n - r0) : 65535;
      if (nts)
        ce_bwd_k<true><<<dim3(gx, (unsigned)nr), dim3(CE_BS), 0, stream()>>>(logits + r0 * c, targets + r0, lse + r0,
                                                                             gloss, dlogits + r0 * c, n, (int)c, vec);
      else
        ce_bwd_k<false><<<dim3(gx, (unsigned)nr), dim3(CE_BS), 0, stream()>>>(logits + r0 * c, targets + r0, lse + r0,
                                                                              gloss, dlogits + r0 * c, n, (int)c, vec);
      if (int rc = check_launch("cross_entropy_bwd")) return rc;
    }
    return OXI_OK;
  }
  if (nts) ce_bwd_k<true><<<dim3(gx, (unsigned)n), dim3(CE_BS), 0, stream()>>>(logits, targets, lse, gloss, dlogits, n, (int)c, vec);
  else ce_bwd_k<false><<<dim3(gx, (unsigned)n), dim3(CE_BS), 0, stream()>>>(logits, targets, lse, gloss, dlogits, n, (int)c, vec);
  return check_launch("cross_entropy_bwd");
}

}  // extern "C"
