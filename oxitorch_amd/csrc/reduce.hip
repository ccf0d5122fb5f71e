// Dim reductions (sum, mean, max, min, argmax, argmin, norm) over strided
// tensors, with the semantics of ReduceKind::reduce_strip
// (crates/oxi-tensor/src/ops.rs:246-285) and Tensor::reduce
// (crates/oxi-tensor/src/lib.rs:519-576).
//
// Kernels:
//   strip-contiguous (reduced dim has stride 1): a wave, or for long strips a
//     block, per strip; lanes read the strip as float4s at any float
//     alignment, four in flight, and the group combines in a fixed tree. Few
//     long strips are cut into parts over the chip, combined by a second
//     launch;
//   strided (any other stride): for sum/mean/norm every output is the
//     reference's own sequential f32 fold over its strip, so the result is
//     bit-identical to it. Many outputs, or few positions: a thread walks the
//     strip of one or four adjacent outputs. Few outputs: a block stages the
//     strips of 16 adjacent outputs through LDS and one lane per output folds
//     them. reduce_route() chooses.
// max/min fold with fmaxf/fminf (NaN ignored, as f32::max/min); argmax/argmin
// keep the first strict winner starting from index 0, so a NaN at index 0
// sticks and later NaNs are ignored. Indices are written as floats.
#include <algorithm>
#include <type_traits>

#include "internal.h"
#include "reduce_route.h"
#include "rowtile.h"

namespace oxi {
namespace {

constexpr int BS = 256;
constexpr int MAXD = OXI_MAX_DIMS;

__device__ __forceinline__ int64_t base_of(const RPlan& p, int64_t e) {
  int64_t off = 0;
  for (int d = p.nd - 1; d >= 0; --d) {
    const int64_t c = e % p.size[d];
    e /= p.size[d];
    off += c * p.st[d];
  }
  return off;
}

// Accumulator state per kind.
template <int K>
struct Acc {
  float v;
  int64_t i;
  __device__ __forceinline__ void init(float first) {
    if constexpr (K == OXI_REDUCE_MAX) v = -__builtin_huge_valf();
    else if constexpr (K == OXI_REDUCE_MIN) v = __builtin_huge_valf();
    else if constexpr (K == OXI_REDUCE_ARGMAX || K == OXI_REDUCE_ARGMIN) v = first;
    else v = 0.f;
    i = 0;
  }
  __device__ __forceinline__ void add(float a, int64_t k) {
    if constexpr (K == OXI_REDUCE_SUM || K == OXI_REDUCE_MEAN) v += a;
    else if constexpr (K == OXI_REDUCE_NORM) v += a * a;
    else if constexpr (K == OXI_REDUCE_MAX) v = fmaxf(v, a);
    else if constexpr (K == OXI_REDUCE_MIN) v = fminf(v, a);
    else if constexpr (K == OXI_REDUCE_ARGMAX) { if (a > v) { v = a; i = k; } }
    else { if (a < v) { v = a; i = k; } }
  }
  __device__ __forceinline__ float result(int64_t len) const {
    if constexpr (K == OXI_REDUCE_MEAN) return v / (float)len;
    else if constexpr (K == OXI_REDUCE_NORM) return sqrtf(v);
    else if constexpr (K == OXI_REDUCE_ARGMAX || K == OXI_REDUCE_ARGMIN) return (float)i;
    else return v;
  }
};

// One thread per output. The loads of STRIDED_U positions issue together and
// are folded in order: the column sums of (512, 50001) 128 -> 19 us (8: 27 us).
constexpr int STRIDED_U = 16;
constexpr int VEC_U = 8;  // the same for four outputs a thread (16: as fast)

template <int K>
__global__ __launch_bounds__(BS) void reduce_strided_k(const float* __restrict__ x, RPlan p, int64_t nout,
                                                       float* __restrict__ out) {
  for (int64_t e = (int64_t)blockIdx.x * BS + threadIdx.x; e < nout; e += (int64_t)gridDim.x * BS) {
    const float* s = x + base_of(p, e);
    Acc<K> a;
    a.init(p.len ? s[0] : 0.f);
    int64_t k = 0;
    for (; k + STRIDED_U <= p.len; k += STRIDED_U) {
      float v[STRIDED_U];
#pragma unroll
      for (int u = 0; u < STRIDED_U; ++u) v[u] = s[(k + u) * p.rst];
#pragma unroll
      for (int u = 0; u < STRIDED_U; ++u) a.add(v[u], k + u);
    }
    for (; k < p.len; ++k) a.add(s[k * p.rst], k);
    out[e] = a.result(p.len);
  }
}

// The state of one lane or group over part of a strip. For
// argmax/argmin it is the first winner among non-NaN values; a NaN at
// position 0 of the strip forces index 0, matching the sequential scan.
template <int K>
struct Part {
  float v;    // arg*: the winner, NaN while there is none
  int64_t i;  // arg*: its position
  static __device__ __forceinline__ Part none() {
    if constexpr (K == OXI_REDUCE_MAX) return {-__builtin_huge_valf(), 0};
    else if constexpr (K == OXI_REDUCE_MIN) return {__builtin_huge_valf(), 0};
    else if constexpr (is_arg(K)) return {__builtin_nanf(""), 0};
    else return {0.f, 0};
  }
  __device__ __forceinline__ void add(float a, int64_t k) {
    if constexpr (K == OXI_REDUCE_SUM || K == OXI_REDUCE_MEAN) v += a;
    else if constexpr (K == OXI_REDUCE_NORM) v += a * a;
    else if constexpr (K == OXI_REDUCE_MAX) v = fmaxf(v, a);
    else if constexpr (K == OXI_REDUCE_MIN) v = fminf(v, a);
    else {
      // not (a <= v): a strict winner, or the first (v is NaN)
      const bool better = !((K == OXI_REDUCE_ARGMAX) ? (a <= v) : (a >= v)) & (a == a);
      v = better ? a : v;
      i = better ? k : i;
    }
  }
  // o may hold positions before or after this one's: a tie goes to the smaller index
  __device__ __forceinline__ void merge(const Part& o) {
    if constexpr (is_fold(K)) v += o.v;
    else if constexpr (K == OXI_REDUCE_MAX) v = fmaxf(v, o.v);
    else if constexpr (K == OXI_REDUCE_MIN) v = fminf(v, o.v);
    else {
      const bool better = !((K == OXI_REDUCE_ARGMAX) ? (o.v <= v) : (o.v >= v)) & (o.v == o.v);
      if (better || (o.v == v && o.i < i)) *this = o;
    }
  }
};

// The state of the lane whose number differs by the mask m.
template <int K>
__device__ __forceinline__ Part<K> part_xor(const Part<K>& a, int m) {
  Part<K> o = Part<K>::none();
  o.v = __shfl_xor(a.v, m, 64);
  if constexpr (is_arg(K)) o.i = __shfl_xor(a.i, m, 64);
  return o;
}

template <int K>
__device__ __forceinline__ float strip_result(const float* s, const Part<K>& a, int64_t len) {
  if constexpr (K == OXI_REDUCE_MEAN) return a.v / (float)len;
  else if constexpr (K == OXI_REDUCE_NORM) return sqrtf(a.v);
  else if constexpr (is_arg(K)) return (s[0] != s[0]) ? 0.f : (float)a.i;
  else return a.v;
}

// Few outputs over long strips: a block owns COLS_C outputs adjacent in
// memory. Its loading threads take COLS_R positions of them at a time
// (coalesced rows of 64 bytes) and store them transposed in LDS, where the
// lanes of one more wave, one per output, fold their strips in order; the next
// positions' loads are in flight meanwhile, and two LDS stages alternate, so
// there is one barrier a stage. What bounds it is that fold, a chain of
// dependent adds of 8 cycles each, which the reference's order fixes (55 us
// for 16384 positions, of the 59 us the 768 columns of such a strip take); max, min and arg* take
// four lanes per output, each a quarter of every stage. VEC: rows of float4s
// (columns a multiple of 4, aligned); else single floats.
constexpr int COLS_NT = COLS_THREADS;
constexpr int COLS_LT = COLS_NT - 64;  // loading threads
constexpr int COLS_R = 512;    // positions a stage
constexpr int COLS_LD = COLS_R + 4;  // floats between outputs in LDS: 16 lanes reading float4s touch 64 distinct banks
constexpr int COLS_F = 32;     // positions a lane has read from LDS ahead of its fold

template <int K, bool VEC>
__global__ __launch_bounds__(COLS_NT) void reduce_cols_k(const float* __restrict__ x, RPlan p, int64_t inner,
                                                         int64_t groups, float* __restrict__ out) {
  constexpr int W = VEC ? 4 : 1;               // floats per load
  constexpr int TPP = COLS_C / W;              // threads per position
  constexpr int PPP = COLS_LT / TPP;           // positions a pass of the block
  constexpr int U = COLS_R / PPP;              // passes a stage
  using V = typename std::conditional<VEC, f4, float>::type;
  __shared__ __align__(16) float tile[2][COLS_C * COLS_LD];
  const int64_t o = blockIdx.x / groups;       // row of outputs
  const int64_t c0 = (blockIdx.x % groups) * COLS_C;
  const int nc = (int)min<int64_t>(COLS_C, inner - c0);  // a multiple of W
  const float* s = x + base_of(p, o * inner + c0);
  const int64_t len = p.len, rst = p.rst;
  if (threadIdx.x < COLS_LT) {
    const int q = threadIdx.x % TPP, r = threadIdx.x / TPP;
    const float* sp = s + min(q * W, nc - W);  // columns past the last output re-read it
    V v[U];
    auto load = [&](int64_t k0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t k = min<int64_t>(k0 + u * PPP + r, len - 1);  // positions past the strip re-read its last
        v[u] = *reinterpret_cast<const V*>(sp + k * rst);  // plain: two blocks share a 128-byte line
      }
    };
    load(0);
    int b = 0;
    for (int64_t k0 = 0; k0 < len; k0 += COLS_R, b ^= 1) {
      float* t = tile[b] + q * W * COLS_LD + r;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if constexpr (VEC) {
#pragma unroll
          for (int j = 0; j < 4; ++j) t[j * COLS_LD + u * PPP] = v[u][j];
        } else {
          t[u * PPP] = v[u];
        }
      }
      if (k0 + COLS_R < len) load(k0 + COLS_R);
      // this stage is written, and the fold of the one before it is done:
      // the next pass may overwrite that one
      __syncthreads();
    }
    return;
  }
  // SUB lanes share an output, lane `sub` folding positions [lo, lo + COLS_R / SUB) of each stage
  constexpr int SUB = is_fold(K) ? 1 : 64 / COLS_C;
  const int lane = threadIdx.x & (COLS_C - 1);
  const int lo = SUB == 1 ? 0 : (int)((threadIdx.x & 63) / COLS_C) * (COLS_R / SUB);
  Part<K> a = Part<K>::none();
  int b = 0;
  for (int64_t k0 = 0; k0 < len; k0 += COLS_R, b ^= 1) {
    __syncthreads();  // the stage is written
    const float* c = tile[b] + lane * COLS_LD + lo;
    const int n = (int)min<int64_t>(COLS_R / SUB, len - k0 - lo);  // <= 0: none of this stage
    f4 fa[COLS_F / 4], fb[COLS_F / 4];
    auto fetch = [&](f4 (&f)[COLS_F / 4], int at) {
      const float* q = c + min(at, COLS_R / SUB - COLS_F);
#pragma unroll
      for (int i = 0; i < COLS_F / 4; ++i) f[i] = *reinterpret_cast<const f4*>(q + 4 * i);
    };
    auto fold = [&](const f4 (&f)[COLS_F / 4], int at) {
#pragma unroll
      for (int i = 0; i < COLS_F; ++i) a.add(f[i / 4][i % 4], k0 + lo + at + i);
    };
    int k = 0;
    fetch(fa, 0);
    // the scheduling barriers keep the next positions' reads above the adds
    for (; k + 2 * COLS_F <= n; k += 2 * COLS_F) {
      fetch(fb, k + COLS_F);
      __builtin_amdgcn_sched_barrier(0);
      fold(fa, k);
      fetch(fa, k + 2 * COLS_F);
      __builtin_amdgcn_sched_barrier(0);
      fold(fb, k + COLS_F);
    }
    for (; k < n; ++k) a.add(c[k], k0 + lo + k);
  }
  if constexpr (SUB > 1) {
#pragma unroll
    for (int m = COLS_C; m < 64; m <<= 1) a.merge(part_xor<K>(a, m));
  }
  const int w = (int)threadIdx.x - COLS_LT;
  if (w < nc) out[o * inner + c0 + w] = strip_result<K>(s + w, a, len);
}

// Four adjacent outputs per thread when they are adjacent in memory (the
// last remaining dim has stride 1): 16-byte loads walk the strip. Same
// sequential fold per output as reduce_strided_k. Not used for arg* kinds.
template <int K>
__global__ __launch_bounds__(BS) void reduce_strided_vec_k(const float* __restrict__ x, RPlan p, int64_t nout4,
                                                           float* __restrict__ out) {
  for (int64_t e4 = (int64_t)blockIdx.x * BS + threadIdx.x; e4 < nout4; e4 += (int64_t)gridDim.x * BS) {
    const float* s = x + base_of(p, e4 * 4);
    f4 a;
    if constexpr (K == OXI_REDUCE_MAX) a = f4{-__builtin_huge_valf(), -__builtin_huge_valf(), -__builtin_huge_valf(), -__builtin_huge_valf()};
    else if constexpr (K == OXI_REDUCE_MIN) a = f4{__builtin_huge_valf(), __builtin_huge_valf(), __builtin_huge_valf(), __builtin_huge_valf()};
    else a = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll VEC_U
    for (int64_t k = 0; k < p.len; ++k) {
      const f4 v = ld_stream(reinterpret_cast<const f4*>(s + k * p.rst));
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if constexpr (K == OXI_REDUCE_SUM || K == OXI_REDUCE_MEAN) a[c] += v[c];
        else if constexpr (K == OXI_REDUCE_NORM) a[c] += v[c] * v[c];
        else if constexpr (K == OXI_REDUCE_MAX) a[c] = fmaxf(a[c], v[c]);
        else a[c] = fminf(a[c], v[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (K == OXI_REDUCE_MEAN) a[c] = a[c] / (float)p.len;
      else if constexpr (K == OXI_REDUCE_NORM) a[c] = sqrtf(a[c]);
    }
    *reinterpret_cast<f4*>(out + e4 * 4) = a;
  }
}

// The state over positions [k0, k1) of strip s, formed by the TPS threads of
// a group (t = 0 .. TPS-1); thread 0 of the group returns it. Float4s at any
// float alignment, CU_LOADS in flight per thread; each of a thread's four
// components folds on its own and they meet in a fixed order.
constexpr int CU_LOADS = 4;

template <int K, int TPS>
__device__ __forceinline__ Part<K> strip_part(const float* __restrict__ s, int64_t k0, int64_t k1, int t,
                                              Part<K>* lds) {
  constexpr int NP = is_arg(K) ? 1 : 4;  // chains per thread (arg*: one, in position order)
  Part<K> a[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) a[j] = Part<K>::none();
  const int64_t n4 = (k1 - k0) >> 2;
  const float* p = s + k0;
  int64_t c = t;
  for (; c + (CU_LOADS - 1) * TPS < n4; c += CU_LOADS * TPS) {
    f4u v[CU_LOADS];
#pragma unroll
    for (int u = 0; u < CU_LOADS; ++u) v[u] = ld_stream(reinterpret_cast<const f4u*>(p + 4 * (c + u * TPS)));
#pragma unroll
    for (int u = 0; u < CU_LOADS; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j % NP].add(v[u][j], k0 + 4 * (c + u * TPS) + j);
  }
  for (; c < n4; c += TPS) {
    const f4u v = ld_stream(reinterpret_cast<const f4u*>(p + 4 * c));
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j % NP].add(v[j], k0 + 4 * c + j);
  }
  if (t < (int)((k1 - k0) & 3)) a[0].add(p[4 * n4 + t], k0 + 4 * n4 + t);
#pragma unroll
  for (int j = 1; j < NP; ++j) a[0].merge(a[j]);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) a[0].merge(part_xor<K>(a[0], m));
  if constexpr (TPS > 64) {
    if ((t & 63) == 0) lds[t >> 6] = a[0];
    __syncthreads();
    if (t == 0)
#pragma unroll
      for (int w = 1; w < TPS / 64; ++w) a[0].merge(lds[w]);
  }
  return a[0];
}

// A strip per group of TPS threads. SHORT (strips of up to WAVE_SHORT_LEN): its
// lanes read single floats.
template <int K, int TPS, bool SHORT = false>
__global__ __launch_bounds__((TPS > BS ? TPS : BS)) void reduce_contig_k(const float* __restrict__ x, RPlan p,
                                                                         int64_t nout, float* __restrict__ out) {
  constexpr int NT = TPS > BS ? TPS : BS;
  __shared__ Part<K> lds[TPS / 64];
  const int t = threadIdx.x % TPS;
  const int64_t e = (int64_t)blockIdx.x * (NT / TPS) + threadIdx.x / TPS;
  if (e >= nout) return;  // TPS > 64: one strip per block, the whole block leaves together
  const float* s = x + base_of(p, e);
  Part<K> a;
  if constexpr (SHORT) {
    static_assert(TPS == 64, "short strips: a wave each");
    a = Part<K>::none();
    for (int k = t; k < (int)p.len; k += TPS) a.add(s[k], k);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) a.merge(part_xor<K>(a, m));
  } else {
    a = strip_part<K, TPS>(s, 0, p.len, t, lds);
  }
  if (t == 0) out[e] = strip_result<K>(s, a, p.len);
}

// Few long strips: block (e, j) leaves the state of positions
// [j * part, (j + 1) * part) of strip e; strip_finish_k merges a strip's
// parts, sums in float64.
template <int K>
__global__ __launch_bounds__(BS) void reduce_parts_k(const float* __restrict__ x, RPlan p, int64_t part, int parts,
                                                     Part<K>* __restrict__ ws) {
  __shared__ Part<K> lds[BS / 64];
  const int64_t e = blockIdx.x / parts;
  const int64_t k0 = (int64_t)(blockIdx.x % parts) * part;
  const Part<K> a = strip_part<K, BS>(x + base_of(p, e), k0, min<int64_t>(k0 + part, p.len), threadIdx.x, lds);
  if (threadIdx.x == 0) ws[blockIdx.x] = a;
}

// A strip's state from its parts', on a wave's lanes t.
template <int K>
__device__ __forceinline__ Part<K> merge_parts(const Part<K>* w, int parts, int t) {
  Part<K> a = Part<K>::none();
  if constexpr (is_fold(K)) {
    double d = 0.0;
    for (int j = t; j < parts; j += 64) d += (double)w[j].v;
    d = wave_sum(d);
    a.v = (float)d;
  } else {
    for (int j = t; j < parts; j += 64) a.merge(w[j]);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) a.merge(part_xor<K>(a, m));
  }
  return a;
}

template <int K>
__global__ __launch_bounds__(64) void strip_finish_k(const float* __restrict__ x, RPlan p, int parts,
                                                     const Part<K>* __restrict__ ws, float* __restrict__ out) {
  const int64_t e = blockIdx.x;
  const Part<K> a = merge_parts<K>(ws + e * parts, parts, threadIdx.x);
  if (threadIdx.x == 0) out[e] = strip_result<K>(x + base_of(p, e), a, p.len);
}

// The same where no workspace can be taken (a captured launch, no memory): a
// block a strip forms its parts' states one after the other, a part to each of
// its four groups of threads, and keeps them in LDS. The results have the bits
// of the two launches; a sum of 200003 floats takes 17 us (10 in two launches),
// of 12.6M 985 (14).
template <int K>
__global__ __launch_bounds__(4 * BS) void reduce_parts_lds_k(const float* __restrict__ x, RPlan p, int64_t part,
                                                             int parts, float* __restrict__ out) {
  __shared__ Part<K> state[SPLIT_MAX_PARTS];
  __shared__ Part<K> lds[4][BS / 64];
  const int64_t e = blockIdx.x;
  const float* s = x + base_of(p, e);
  const int t = threadIdx.x % BS, group = threadIdx.x / BS;
  for (int j0 = 0; j0 < parts; j0 += 4) {  // every thread makes every round: strip_part has a barrier
    const int j = j0 + group;
    const int64_t k0 = min<int64_t>((int64_t)j * part, p.len);  // past the last part: nothing
    const Part<K> a = strip_part<K, BS>(s, k0, min<int64_t>(k0 + part, p.len), t, lds[group]);
    if (t == 0 && j < parts) state[j] = a;
    __syncthreads();  // lds is free again
  }
  if (threadIdx.x < 64) {
    const Part<K> a = merge_parts<K>(state, parts, threadIdx.x);
    if (threadIdx.x == 0) out[e] = strip_result<K>(s, a, p.len);
  }
}

// Whether the library stream is being captured into a graph: a launch that
// needs a workspace then takes the kernel without one (the block would go back
// to the allocator when the call returns, and be written again by a replay).
bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

template <int K>
int launch(const float* x, const RPlan& p, int64_t nout, float* out) {
  hipStream_t s = stream();
  const ReduceRoute r = reduce_route(K, p, nout, x, out, cu_count());
  if (r.kernel == ReduceKernel::Parts) {
    if (!capturing(s)) {
      Workspace ws(sizeof(Part<K>) * (size_t)r.blocks);
      if (ws.p) {
        reduce_parts_k<K><<<dim3((unsigned)r.blocks), dim3(BS), 0, s>>>(x, p, r.part, (int)r.parts, ws.as<Part<K>>());
        if (int rc = check_launch("reduce")) return rc;
        strip_finish_k<K><<<dim3((unsigned)nout), dim3(64), 0, s>>>(x, p, (int)r.parts, ws.as<Part<K>>(), out);
        return check_launch("reduce_finish");
      }
    }
    reduce_parts_lds_k<K><<<dim3((unsigned)nout), dim3(4 * BS), 0, s>>>(x, p, r.part, (int)r.parts, out);
    return check_launch("reduce");
  }
  const dim3 g((unsigned)r.blocks);
  switch (r.kernel) {
    case ReduceKernel::Strips:
      if (p.len <= WAVE_SHORT_LEN) reduce_contig_k<K, 64, true><<<g, dim3(BS), 0, s>>>(x, p, nout, out);
      else if (r.threads == 64) reduce_contig_k<K, 64><<<g, dim3(BS), 0, s>>>(x, p, nout, out);
      else if (r.threads == 256) reduce_contig_k<K, 256><<<g, dim3(256), 0, s>>>(x, p, nout, out);
      else reduce_contig_k<K, 1024><<<g, dim3(1024), 0, s>>>(x, p, nout, out);
      break;
    case ReduceKernel::Cols:
      if (r.vec) reduce_cols_k<K, true><<<g, dim3(COLS_NT), 0, s>>>(x, p, r.inner, r.groups, out);
      else reduce_cols_k<K, false><<<g, dim3(COLS_NT), 0, s>>>(x, p, r.inner, r.groups, out);
      break;
    case ReduceKernel::Vec:
      if constexpr (!is_arg(K)) reduce_strided_vec_k<K><<<g, dim3(BS), 0, s>>>(x, p, nout / 4, out);
      break;
    default:
      reduce_strided_k<K><<<g, dim3(BS), 0, s>>>(x, p, nout, out);
  }
  return check_launch("reduce");
}

}  // namespace
}  // namespace oxi

using namespace oxi;

extern "C" {

int oxi_reduce(int kind, const float* x, const int64_t* xs, const int64_t* shape, int ndim, int dim, float* out) {
  if (kind < OXI_REDUCE_SUM || kind > OXI_REDUCE_NORM) return fail(OXI_INVALID_ARGUMENT, "unknown reduction kind %d", kind);
  if (ndim < 1 || ndim > MAXD) return fail(OXI_INVALID_ARGUMENT, "reduce: rank %d outside [1, %d]", ndim, MAXD);
  if (dim < 0 || dim >= ndim) return fail(OXI_INVALID_ARGUMENT, "reduce: dim %d out of range for rank %d", dim, ndim);
  if (!shape || !xs) return fail(OXI_INVALID_ARGUMENT, "reduce: NULL shape/strides");
  RPlan p;
  p.nd = 0;
  int64_t nout = 1;
  int64_t total = 1;
  for (int d = 0; d < ndim; ++d) {
    if (shape[d] < 0) return fail(OXI_INVALID_ARGUMENT, "reduce: negative dim size");
    if (shape[d] && total > (((int64_t)1 << 60) / shape[d]))
      return fail(OXI_INVALID_ARGUMENT, "reduce: element count exceeds the kernel limits");
    total *= shape[d];
    if (d == dim) continue;
    p.size[p.nd] = shape[d];
    p.st[p.nd] = xs[d];
    ++p.nd;
    nout *= shape[d];
  }
  p.len = shape[dim];
  p.rst = xs[dim];
  if (p.len == 0) {
    if (kind == OXI_REDUCE_ARGMAX || kind == OXI_REDUCE_ARGMIN)
      return fail(OXI_INVALID_ARGUMENT, "cannot compute argmax/argmin over a zero-length dim");
    if (kind == OXI_REDUCE_MAX || kind == OXI_REDUCE_MIN)
      return fail(OXI_INVALID_ARGUMENT, "cannot compute max/min over a zero-length dim");
  }
  if (nout == 0) return OXI_OK;
  if (!out || (!x && p.len)) return fail(OXI_INVALID_ARGUMENT, "reduce: NULL tensor pointer");
  OXI_CHECK_INIT();
  if (p.len == 0) return oxi_fill(out, nout, 0.f);
  simplify(p);
  switch (kind) {
    case OXI_REDUCE_SUM: return launch<OXI_REDUCE_SUM>(x, p, nout, out);
    case OXI_REDUCE_MEAN: return launch<OXI_REDUCE_MEAN>(x, p, nout, out);
    case OXI_REDUCE_MAX: return launch<OXI_REDUCE_MAX>(x, p, nout, out);
    case OXI_REDUCE_MIN: return launch<OXI_REDUCE_MIN>(x, p, nout, out);
    case OXI_REDUCE_ARGMAX: return launch<OXI_REDUCE_ARGMAX>(x, p, nout, out);
    case OXI_REDUCE_ARGMIN: return launch<OXI_REDUCE_ARGMIN>(x, p, nout, out);
    default: return launch<OXI_REDUCE_NORM>(x, p, nout, out);
  }
}

}  // extern "C"
