// linear.hip - y = x W^T for few rows of x, on gfx950 MFMA.
//
// The projections of a short prompt or of a follow-up of a few tokens read
// each weight once for a handful of rows: they are bound by that read and by
// their launches. A library GEMM costs ~17 us of host time per call here
// (its choice of kernel is made again every time), more than the kernel runs.
//
// A workgroup owns 16 rows of W (16 gate and the 16 matching up rows in the
// SwiGLU form) and up to 64 rows of x; its 8 wavefronts split K in steps of
// 32, so that even N = 1024 keeps 512 wavefronts loading. Per step a lane
// loads 16 bytes of its W row and of its rows of x straight into MFMA
// operands (16x16x32: row lane % 16, k = 8 (lane / 16) ..), several steps
// ahead; nothing is shared, so nothing is staged in LDS. The wavefronts'
// fp32 sums are added through LDS in a fixed order, rounded once and stored.
// The SwiGLU form rounds gate and up first, as the GEMM's output would be.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "internal.h"
#include "silu.h"

namespace ttcd {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

template <typename T>
struct Vec8;
template <>
struct Vec8<__bf16> {
  typedef bf16x8 t;
};
template <>
struct Vec8<_Float16> {
  typedef f16x8 t;
};

constexpr int kLinWaves = 8;
constexpr int kStep = 32;     // k per MFMA
constexpr int kUnroll = 4;    // steps whose loads are in flight together

// MT: tiles of 16 rows of x; GLU: the SwiGLU form (w holds 2 N rows).
template <typename T, int MT, bool GLU>
__global__ __launch_bounds__(kLinWaves * 64) void linear_rows_kernel(LinearArgs a) {
  typedef typename Vec8<T>::t v8;
  constexpr int NT = GLU ? 2 : 1;
  __shared__ float part[kLinWaves][NT][MT][16][17];  // [wave][tile][m tile][n][m]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * MT);
  const int r = lane & 15, kq = (lane >> 4) * 8;

  // rows past the end read the last one and are not stored
  const T* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    wp[t] = static_cast<const T*>(a.w) +
            ((int64_t)t * a.N + min(n0 + r, a.N - 1)) * a.K + kq;
  const T* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
    xp[t] = static_cast<const T*>(a.x) + (int64_t)min(m0 + 16 * t + r, a.M - 1) * a.x_st + kq;

  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = a.K / kStep;
  for (int s0 = wave; s0 < steps; s0 += kLinWaves * kUnroll) {
    v8 wv[kUnroll][NT], xv[kUnroll][MT];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      // a step past the end re-reads the wavefront's first one, unused
      const int s = s0 + u * kLinWaves;
      const int64_t k = (int64_t)(s < steps ? s : s0) * kStep;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        wv[u][t] = __builtin_nontemporal_load(reinterpret_cast<const v8*>(wp[t] + k));
#pragma unroll
      for (int t = 0; t < MT; ++t) xv[u][t] = *reinterpret_cast<const v8*>(xp[t] + k);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      if (s0 + u * kLinWaves < steps) {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
          for (int j = 0; j < MT; ++j) acc[i][j] = mfma16(wv[u][i], xv[u][j], acc[i][j]);
      }
    }
  }
  // accumulator element e: W row 4 (lane / 16) + e, x row lane % 16
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[wave][i][j][4 * (lane >> 4) + e][r] = acc[i][j][e];
  __syncthreads();
  T* y = static_cast<T*>(a.y);
  for (int i = threadIdx.x; i < 256 * MT; i += kLinWaves * 64) {
    const int n = i & 15, m = (i >> 4) & 15, j = i >> 8;
    float s[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      s[t] = 0.f;
#pragma unroll
      for (int w = 0; w < kLinWaves; ++w) s[t] += part[w][t][j][n][m];
    }
    if (n0 + n < a.N && m0 + 16 * j + m < a.M) {
      float v = s[0];
      if constexpr (GLU)
        v = silu_mul(static_cast<float>(round_to<T>(s[0])),
                     static_cast<float>(round_to<T>(s[NT - 1])));
      y[(int64_t)(m0 + 16 * j + m) * a.N + n0 + n] = round_to<T>(v);
    }
  }
}

template <typename T, int MT>
hipError_t launch_mt(const LinearArgs& a, hipStream_t st) {
  const dim3 grid((a.N + 15) / 16, (a.M + 16 * MT - 1) / (16 * MT));
  if (a.glu)
    hipLaunchKernelGGL((linear_rows_kernel<T, MT, true>), grid, dim3(kLinWaves * 64), 0, st, a);
  else
    hipLaunchKernelGGL((linear_rows_kernel<T, MT, false>), grid, dim3(kLinWaves * 64), 0, st, a);
  return hipGetLastError();
}

// As many rows of x per workgroup as leave 256 workgroups: a workgroup's time
// grows with its rows (its loads of x), not with its neighbours'.
template <typename T>
hipError_t launch_typed(const LinearArgs& a, hipStream_t st) {
  const int64_t cols = (a.N + 15) / 16;
  auto fills = [&](int mt) { return cols * ((a.M + 16 * mt - 1) / (16 * mt)) >= 256; };
  if (a.M > 32 && fills(4)) return launch_mt<T, 4>(a, st);
  if (a.M > 16 && fills(2)) return launch_mt<T, 2>(a, st);
  return launch_mt<T, 1>(a, st);
}

}  // namespace

hipError_t launch_linear_rows(const LinearArgs& a, Elem dtype, hipStream_t stream) {
  return dtype == Elem::BF16 ? launch_typed<__bf16>(a, stream) : launch_typed<_Float16>(a, stream);
}

}  // namespace ttcd
