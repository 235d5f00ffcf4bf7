// conv.hip - chunk-local causal depthwise conv on the (N, C, D) layout for
// gfx950. Replaces the Triton kernel _causal_dwconv_fwd
// (profiling/fused_conv.py:24-48): y[n,c,d] = sum_j w[d,j] * x[n,c-(K-1)+j,d]
// with left zero padding inside each chunk, fp32 accumulation in tap order
// j = 0..K-1 (acc = fma(x, w, acc) from acc = +0), one RNE rounding to the
// input dtype.
//
// The op is HBM-bound (one read of x, one write of y), so there is no MFMA
// here. Each thread owns 16 bytes along D (8 bf16 channels) and a run of R
// consecutive rows along C, and the K-1 previous rows stay in registers as a
// sliding window. For K <= 8 (dwconv_halo_kernel) a wavefront holds 16
// groups along D of 4 consecutive runs, and each run's K-1 halo rows come
// from the run below it through a lane shuffle, so x is read (4R + K - 1) /
// 4R times. (A halo re-read from memory by every run misses L2 as often as
// not: it is requested while the neighbouring run fetches the same rows,
// which cost 25 % more HBM reads at R = 16.) y is written with non-temporal
// stores: it is consumed by the next op, not by this kernel.
//
// Rows that are not 16-byte aligned (D not a multiple of a group, or a base
// address off it) take the same kernel with accesses of element alignment,
// the last group of a row moved back to end with it. K > 8 takes
// dwconv_taps_kernel, which slides over the taps instead. Small calls and rows
// shorter than one group take dwconv_scalar_kernel, one thread per output.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "internal.h"

namespace ttcd {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename X>
struct Cvt;
template <>
struct Cvt<__bf16> {
  __device__ static float to_f(__bf16 v) { return static_cast<float>(v); }
  __device__ static __bf16 from_f(float v) { return static_cast<__bf16>(v); }
};
template <>
struct Cvt<_Float16> {
  __device__ static float to_f(_Float16 v) { return static_cast<float>(v); }
  // The empty asm pins the fp32 sum in a register first. Without it the compiler
  // fuses the last tap's fma with this conversion (v_fma_mix{lo,hi}_f16), which
  // rounds once from the exact value instead of fp32-then-fp16 as the reference
  // conv does, and about one output in 8K differs in its last bit.
  __device__ static _Float16 from_f(float v) {
    __asm__("" : "+v"(v));
    return static_cast<_Float16>(v);
  }
};
template <>
struct Cvt<float> {
  __device__ static float to_f(float v) { return v; }
  __device__ static float from_f(float v) { return v; }
};

template <typename X>
union Pack16 {
  static constexpr int N = 16 / sizeof(X);
  u32x4 raw;
  X e[N];
};

// 16 bytes at an address aligned to 16 bytes (AL) or only to an element.
template <bool AL, typename X>
__device__ __forceinline__ u32x4 load16(const X* p) {
  if constexpr (AL) return *reinterpret_cast<const u32x4*>(p);
  u32x4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}
// The last n of the 16 bytes' elements (n == V: all; fewer only when not AL).
template <bool AL, typename X>
__device__ __forceinline__ void store16(X* p, const Pack16<X>& v, int n) {
  if constexpr (AL) {
    __builtin_nontemporal_store(v.raw, reinterpret_cast<u32x4*>(p));
  } else if (n == Pack16<X>::N) {
    __builtin_memcpy(p, &v.raw, 16);
  } else {
    Pack16<X> t = v;
    __asm__ volatile("" : "+v"(t.raw));  // keeps the whole store above one access
#pragma unroll
    for (int e = 0; e < Pack16<X>::N; ++e)
      if (e >= Pack16<X>::N - n) p[e] = t.e[e];
  }
}

// The channel group dg of a row of D channels: its first channel, moved back
// for a last group that would pass the row's end, and how many of its
// channels are its own (the last ones).
template <int V>
__device__ __forceinline__ int group_of(int dg, int D, int* own) {
  const int d0 = dg * V;
  *own = min(V, D - d0);
  return min(d0, D - V);
}

constexpr int kRows = 16;  // rows of C per thread

// Shared-halo layout (K <= kRows + 1): a wavefront owns 16 consecutive
// 16-byte groups along D (lane % 16) of 4 consecutive runs along C (lane /
// 16), so each row access is four contiguous 256-byte pieces. The K-1 halo
// rows of run g are the last rows of run g-1, taken from the lanes 16 below
// with a lane shuffle; only the first run of a wavefront reads its halo from
// memory, so x is read (kRows * 4 + K - 1) / (kRows * 4) times instead of
// (kRows + K - 1) / kRows.
template <typename X, typename W, int K, bool AL>
__global__ __launch_bounds__(256) void dwconv_halo_kernel(const X* __restrict__ x,
                                                          const W* __restrict__ w,
                                                          X* __restrict__ y, int64_t N, int C,
                                                          int D, int nseg) {
  static_assert(K - 1 <= kRows, "the halo must lie within the previous run");
  constexpr int V = Pack16<X>::N;
  const int ngroups = (D + V - 1) / V;
  const int ntile = (ngroups + 15) / 16;
  const int nquad = (nseg + 3) / 4;
  const int lane = threadIdx.x & 63;
  // one wavefront per (n, quad of runs, 16-group tile); whole wavefronts leave
  const int64_t wid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t total = N * nquad * (int64_t)ntile;
  if (wid >= total) return;
  const int tile = (int)(wid % ntile);
  const int64_t rest = wid / ntile;
  const int quad = (int)(rest % nquad);
  const int64_t n = rest / nquad;
  const int g = lane >> 4;
  const int dg = tile * 16 + (lane & 15);
  const bool col_ok = dg < ngroups;
  int own;
  const int d0 = group_of<V>(col_ok ? dg : 0, D, &own);  // idle lanes read a valid group, store nothing
  const int c0 = (quad * 4 + g) * kRows;
  const int rows = col_ok ? max(0, min(kRows, C - c0)) : 0;

  float wr[K][V];
#pragma unroll
  for (int e = 0; e < V; ++e)
#pragma unroll
    for (int j = 0; j < K; ++j) wr[j][e] = Cvt<W>::to_f(w[(int64_t)(d0 + e) * K + j]);

  const X* xb = x + n * C * (int64_t)D + d0;
  X* yb = y + n * C * (int64_t)D + d0;

  Pack16<X> in[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    in[r].raw = u32x4{0u, 0u, 0u, 0u};
    if (r < rows) in[r].raw = load16<AL>(xb + (int64_t)(c0 + r) * D);
  }

  // win[t] holds row c - (K-1) + t for the row c being produced. Every lane
  // takes part in the shuffles; run g > 0 has a full run g-1 below it.
  float win[K][V];
#pragma unroll
  for (int t = 0; t < K - 1; ++t) {
    Pack16<X> p;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      p.raw[q] = (uint32_t)__shfl_up((int)in[kRows - (K - 1) + t].raw[q], 16, 64);
    if (g == 0) {
      const int c = c0 - (K - 1) + t;
      p.raw = u32x4{0u, 0u, 0u, 0u};
      if (c >= 0 && rows > 0) p.raw = load16<AL>(xb + (int64_t)c * D);
    }
#pragma unroll
    for (int e = 0; e < V; ++e) win[t][e] = Cvt<X>::to_f(p.e[e]);
  }

#pragma unroll
  for (int r = 0; r < kRows; ++r) {
#pragma unroll
    for (int e = 0; e < V; ++e) win[K - 1][e] = Cvt<X>::to_f(in[r].e[e]);
    Pack16<X> out;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < K; ++j) acc = fmaf(win[j][e], wr[j][e], acc);
      out.e[e] = Cvt<X>::from_f(acc);
    }
    if (r < rows) store16<AL>(yb + (int64_t)(c0 + r) * D, out, own);
#pragma unroll
    for (int t = 0; t < K - 1; ++t)
#pragma unroll
      for (int e = 0; e < V; ++e) win[t][e] = win[t + 1][e];
  }
}

// Any K (<= 64): a thread owns one group along D of kTapRows rows and slides
// over the taps, one row loaded per tap, so each row is read (kTapRows + K -
// 1) / kTapRows times (through the cache: the rows above are its neighbours').
constexpr int kTapRows = 8;

template <typename X, typename W, bool AL>
__global__ __launch_bounds__(256) void dwconv_taps_kernel(const X* __restrict__ x,
                                                          const W* __restrict__ w,
                                                          X* __restrict__ y, int64_t N, int C,
                                                          int D, int K, int nseg) {
  constexpr int V = Pack16<X>::N;
  const int ngroups = (D + V - 1) / V;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= N * nseg * (int64_t)ngroups) return;
  const int dg = (int)(gid % ngroups);
  const int64_t rest = gid / ngroups;
  const int c0 = (int)(rest % nseg) * kTapRows;
  const int64_t n = rest / nseg;
  int own;
  const int d0 = group_of<V>(dg, D, &own);
  const X* xb = x + n * C * (int64_t)D + d0;
  X* yb = y + n * C * (int64_t)D + d0;
  const W* wb = w + (int64_t)d0 * K;
  auto row = [&](int c) {
    Pack16<X> p;
    p.raw = u32x4{0u, 0u, 0u, 0u};
    if (c >= 0 && c < C) p.raw = load16<AL>(xb + (int64_t)c * D);
    return p;
  };

  // win[(j + r) % kTapRows] is the row of output r at tap j
  Pack16<X> win[kTapRows];
  float acc[kTapRows][V];
#pragma unroll
  for (int r = 0; r < kTapRows; ++r) {
    if (r < kTapRows - 1) win[r] = row(c0 - (K - 1) + r);
#pragma unroll
    for (int e = 0; e < V; ++e) acc[r][e] = 0.f;
  }
  for (int j0 = 0; j0 < K; j0 += kTapRows) {
#pragma unroll
    for (int i = 0; i < kTapRows; ++i) {
      const int j = j0 + i;
      if (j >= K) break;
      win[(i + kTapRows - 1) % kTapRows] = row(c0 - (K - 1) + j + kTapRows - 1);
      float wj[V];
#pragma unroll
      for (int e = 0; e < V; ++e) wj[e] = Cvt<W>::to_f(wb[(int64_t)e * K + j]);
#pragma unroll
      for (int r = 0; r < kTapRows; ++r)
#pragma unroll
        for (int e = 0; e < V; ++e)
          acc[r][e] = fmaf(Cvt<X>::to_f(win[(i + r) % kTapRows].e[e]), wj[e], acc[r][e]);
    }
  }
#pragma unroll
  for (int r = 0; r < kTapRows; ++r) {
    Pack16<X> out;
#pragma unroll
    for (int e = 0; e < V; ++e) out.e[e] = Cvt<X>::from_f(acc[r][e]);
    if (c0 + r < C) store16<AL>(yb + (int64_t)(c0 + r) * D, out, own);
  }
}

// Any K, any D: one thread per output element, taps re-read through the cache.
// Same fixed accumulation order as the vector kernels.
template <typename X, typename W>
__global__ __launch_bounds__(256) void dwconv_scalar_kernel(const X* __restrict__ x,
                                                            const W* __restrict__ w,
                                                            X* __restrict__ y, int64_t N, int C,
                                                            int D, int K) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = N * C * (int64_t)D;
  if (gid >= total) return;
  const int d = (int)(gid % D);
  const int64_t rest = gid / D;
  const int c = (int)(rest % C);
  const int64_t n = rest / C;
  const X* xb = x + n * C * (int64_t)D + d;
  float acc = 0.f;
  for (int j = 0; j < K; ++j) {
    const int src = c - (K - 1) + j;
    const float xv = src >= 0 ? Cvt<X>::to_f(xb[(int64_t)src * D]) : 0.f;
    acc = fmaf(xv, Cvt<W>::to_f(w[(int64_t)d * K + j]), acc);
  }
  y[gid] = Cvt<X>::from_f(acc);
}

template <typename X, typename W, int K, bool AL>
hipError_t launch_halo(const void* x, const void* w, void* y, int64_t N, int C, int D,
                       hipStream_t st) {
  constexpr int V = Pack16<X>::N;
  const int nseg = (C + kRows - 1) / kRows;
  const int64_t waves = N * ((nseg + 3) / 4) * (int64_t)(((D + V - 1) / V + 15) / 16);
  const int64_t blocks = (waves * 64 + 255) / 256;
  hipLaunchKernelGGL((dwconv_halo_kernel<X, W, K, AL>), dim3((unsigned)blocks), dim3(256), 0, st,
                     static_cast<const X*>(x), static_cast<const W*>(w), static_cast<X*>(y), N,
                     C, D, nseg);
  return hipGetLastError();
}

template <typename X, typename W, bool AL>
hipError_t launch_vec(const void* x, const void* w, void* y, int64_t N, int C, int D, int K,
                      hipStream_t st) {
  switch (K) {
    case 1: return launch_halo<X, W, 1, AL>(x, w, y, N, C, D, st);
    case 2: return launch_halo<X, W, 2, AL>(x, w, y, N, C, D, st);
    case 3: return launch_halo<X, W, 3, AL>(x, w, y, N, C, D, st);
    case 4: return launch_halo<X, W, 4, AL>(x, w, y, N, C, D, st);
    case 5: return launch_halo<X, W, 5, AL>(x, w, y, N, C, D, st);
    case 6: return launch_halo<X, W, 6, AL>(x, w, y, N, C, D, st);
    case 7: return launch_halo<X, W, 7, AL>(x, w, y, N, C, D, st);
    case 8: return launch_halo<X, W, 8, AL>(x, w, y, N, C, D, st);
    default: break;
  }
  constexpr int V = Pack16<X>::N;
  const int nseg = (C + kTapRows - 1) / kTapRows;
  const int64_t threads = N * nseg * (int64_t)((D + V - 1) / V);
  hipLaunchKernelGGL((dwconv_taps_kernel<X, W, AL>), dim3((unsigned)((threads + 255) / 256)),
                     dim3(256), 0, st, static_cast<const X*>(x), static_cast<const W*>(w),
                     static_cast<X*>(y), N, C, D, K, nseg);
  return hipGetLastError();
}

// Up to this many outputs the one-thread-per-output kernel is the faster: its
// threads fill more CUs and each waits for one short chain of loads, where a
// run of 16 rows waits for its whole run. Kernel time, scalar / vector (us),
// bf16: 256 x 256 K = 5 3.4 / 5.2, 1024 x 512 K = 5 4.8 / 5.8 and K = 9 6.0 /
// 7.6, 2048 x 1024 K = 5 11.3 / 6.1, 4096 x 2048 K = 9 59 / 16; rows off
// alignment 512 x 255 3.5 / 8.3, 2048 x 2047 K = 5 20 / 9.3; f32 1024 x 512
// K = 5 4.6 / 4.8. Large, before there was a vector form: 20480 x 1537 K = 5
// 205 -> 30, 32768 x 2560 K = 9 835 -> 140.
constexpr int64_t kScalarOutputs = int64_t(1) << 19;

template <typename X, typename W>
hipError_t launch_typed(const void* x, const void* w, void* y, int64_t N, int C, int D, int K,
                        hipStream_t st) {
  constexpr int V = Pack16<X>::N;
  const bool aligned = (D % V) == 0 && (reinterpret_cast<uintptr_t>(x) % 16) == 0 &&
                       (reinterpret_cast<uintptr_t>(y) % 16) == 0;
  const int64_t total = N * C * (int64_t)D;
  if (total > kScalarOutputs && aligned) return launch_vec<X, W, true>(x, w, y, N, C, D, K, st);
  if (total > kScalarOutputs && D >= V) return launch_vec<X, W, false>(x, w, y, N, C, D, K, st);
  const int64_t blocks = (total + 255) / 256;
  hipLaunchKernelGGL((dwconv_scalar_kernel<X, W>), dim3((unsigned)blocks), dim3(256), 0, st,
                     static_cast<const X*>(x), static_cast<const W*>(w), static_cast<X*>(y), N,
                     C, D, K);
  return hipGetLastError();
}

template <typename X>
hipError_t launch_w(const void* x, const void* w, void* y, int64_t N, int C, int D, int K,
                    Elem wt, hipStream_t st) {
  switch (wt) {
    case Elem::BF16: return launch_typed<X, __bf16>(x, w, y, N, C, D, K, st);
    case Elem::F16: return launch_typed<X, _Float16>(x, w, y, N, C, D, K, st);
    default: return launch_typed<X, float>(x, w, y, N, C, D, K, st);
  }
}

}  // namespace

hipError_t launch_dwconv(const void* x, const void* w, void* y, int64_t N, int C, int D, int K,
                         Elem xt, Elem wt, hipStream_t stream) {
  switch (xt) {
    case Elem::BF16: return launch_w<__bf16>(x, w, y, N, C, D, K, wt, stream);
    case Elem::F16: return launch_w<_Float16>(x, w, y, N, C, D, K, wt, stream);
    default: return launch_w<float>(x, w, y, N, C, D, K, wt, stream);
  }
}

}  // namespace ttcd
