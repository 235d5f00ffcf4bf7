// linear.hip - y = x W^T for few rows of x, on gfx950 MFMA.
//
// The projections of a short prompt or of a follow-up of a few tokens read
// each weight once for a handful of rows: they are bound by that read and by
// their launches. A library GEMM costs ~19 us of host time per call here
// (its choice of kernel is made again every time), more than the kernel runs.
// Which of the two a call takes is decided by shape in linear.py (_pays).
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

// ---------------------------------------------------------------------------
// More rows: 64 x 64 tiles through LDS. 4 wavefronts, each 32 rows of W by 32
// of x (32x32x16 MFMA; in the SwiGLU form of 64 gate and the 64 matching up
// rows), K in steps of 64, a ring of 3 steps filled by global -> LDS DMA 2
// steps ahead. A row of a step is 128 bytes, 8 chunks of 16, chunk c stored at
// c ^ (row & 7), so the 32 lanes of an operand read touch all banks evenly.
// Small tiles, because a call of a few hundred rows has few: 4096 x 1024, 300
// rows, is 320 of them. A step then moves 16 KiB into LDS and 32 KiB out for
// 16 MFMAs, and that LDS traffic bounds it (0.26 us a step; a 4-step ring is no
// faster). Kernel / library (us, weights not in a cache): 4096 x 1024 128 rows
// 7.7 / 12.5, 512 rows 11.2 / 13.1; 6144 x 1024 300 rows 11.2 / 13.3, 512 rows
// 16.4 / 15.2; 1024 x 3072 128 rows 16.4 / 9.8, 512 rows 15.9 / 15.1. The last
// shape's chain of 24 steps on 32 to 128 CUs is what the library shortens by
// splitting K over workgroups.
constexpr int kTileRows = 64;
constexpr int kTileK = 64;
constexpr int kRowBytes = kTileK * 2;
constexpr int kOperandBytes = kTileRows * kRowBytes;  // 8 KiB

#define LDS_AS __attribute__((address_space(3)))

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 16 bytes per lane from base + voff into LDS bytes [lds, lds + 1024) (wave-
// uniform base and lds); its completion is waited for with vmcnt by hand.
__device__ __forceinline__ void dma16(const void* base, uint32_t voff, uint32_t lds) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  const uint64_t bs = (uint64_t)lo | ((uint64_t)hi << 32);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2"
               :
               : "v"(voff), "s"(__builtin_amdgcn_readfirstlane(lds)), "s"(bs)
               : "memory", "m0");
}
#pragma clang diagnostic pop

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// KS: groups of 4 wavefronts that take the steps in turn, each with a ring of
// its own, their sums added through LDS (group 1's to group 0's).
template <typename T, bool GLU, int KS>
__global__ __launch_bounds__(256 * KS) void linear_tile_kernel(LinearArgs a) {
  typedef typename Vec8<T>::t v8;
  constexpr int NT = GLU ? 2 : 1;
  constexpr int NOP = NT + 1;  // operands per stage: W tiles, then x
  constexpr int LOADS = NOP * kOperandBytes / 4096;  // 16-byte loads per lane and step
  constexpr int ST = 3;  // 48 to 144 KiB of rings
  constexpr int RING = ST * NOP * kOperandBytes;
  __shared__ __attribute__((aligned(1024))) char smem[KS * RING];
  const int lane = threadIdx.x & 63;
  const int group = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
  const int n0 = blockIdx.x * kTileRows, m0 = blockIdx.y * kTileRows;
  LDS_AS char* lds = (LDS_AS char*)smem + group * RING;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

  // The lane's i-th load of a step: operand i / 2, row and chunk of LDS slot
  // (wave + 4 (i % 2)) * 64 + lane. Rows past the end read the last one.
  uint32_t voff[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int slot = (wave + 4 * (i & 1)) * 64 + lane;
    const int row = slot >> 3, ch = (slot & 7) ^ (row & 7);
    const int64_t r = i / 2 < NT ? (int64_t)min(n0 + row, a.N - 1) * a.K
                                 : (int64_t)min(m0 + row, a.M - 1) * a.x_st;
    voff[i] = (uint32_t)(r * 2 + ch * 16);
  }
  const char* const wb = static_cast<const char*>(a.w);
  const char* const xb = static_cast<const char*>(a.x);
  // this group's step s is step s * KS + group of K; the groups make the same
  // number of turns (barriers), the last of which may be empty for group 1
  const int all = a.K / kTileK;
  const int steps = (all - group + KS - 1) / KS, turns = (all + KS - 1) / KS;
  auto fetch = [&](int s) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + (s % ST) * (NOP * kOperandBytes) + wave * 1024;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int op = i / 2;
      const char* base = op < NT ? wb + (int64_t)op * a.N * a.K * 2 : xb;
      dma16(base + ((int64_t)s * KS + group) * kRowBytes, voff[i], dst + op * kOperandBytes + (i & 1) * 4096);
    }
  };
#pragma unroll
  for (int s = 0; s < ST - 1; ++s)
    if (s < steps) fetch(s);

  const int wn = wave & 1, wm = wave >> 1;
  const int row = lane & 31, half = lane >> 5;
  const uint32_t sw = (uint32_t)(row & 7);
  const uint32_t wrow = (uint32_t)((wn * 32 + row) * kRowBytes);
  const uint32_t xrow = (uint32_t)(NT * kOperandBytes + (wm * 32 + row) * kRowBytes);
  f32x16 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x16{};
  for (int s = 0; s < turns; ++s) {
    // step s has landed when only the later steps' loads are outstanding; the
    // barrier also ends every read of the stage that step s + ST - 1 replaces
    if (s + ST - 2 < steps)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((ST - 2) * LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    if (s + ST - 1 < steps) fetch(s + ST - 1);
    if (KS > 1 && s >= steps) break;  // the last turn
    const LDS_AS char* st = lds + (s % ST) * (NOP * kOperandBytes);
#pragma unroll
    for (int ks = 0; ks < kTileK / 16; ++ks) {
      const uint32_t ch = (uint32_t)((2 * ks + half) ^ sw) * 16;
      const v8 xv = *(const LDS_AS v8*)(st + xrow + ch);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const v8 wv = *(const LDS_AS v8*)(st + t * kOperandBytes + wrow + ch);
        acc[t] = mfma32(wv, xv, acc[t]);
      }
    }
    // the reads are done before the next step's barrier lets their stage go
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  if constexpr (KS > 1) {
    // [tile][element][lane of the 4 wavefronts], over the rings: every read of
    // them is done
    static_assert(KS == 2 && NT * 16 * 256 * 4 <= KS * RING, "sums fit over the rings");
    float* part = reinterpret_cast<float*>(smem);
    const int at = wave * 64 + lane;
    __syncthreads();
    if (group == 1) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) part[(t * 16 + e) * 256 + at] = acc[t][e];
    }
    __syncthreads();
    if (group == 1) return;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[t][e] += part[(t * 16 + e) * 256 + at];
  }
  // accumulator element e: W row 8 (e / 4) + 4 half + e % 4, x row lane % 32
  const int m = m0 + wm * 32 + row;
  if (m >= a.M) return;
  T* y = static_cast<T*>(a.y) + (int64_t)m * a.N;
  const bool wide = a.N % 4 == 0 && (reinterpret_cast<uintptr_t>(a.y) & 7u) == 0;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int n = n0 + wn * 32 + 8 * g + 4 * half;
    union {
      T e[4];
      u32x2 raw;
    } v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float f = acc[0][4 * g + e];
      if constexpr (GLU)
        f = silu_mul(static_cast<float>(round_to<T>(f)),
                     static_cast<float>(round_to<T>(acc[NT - 1][4 * g + e])));
      v.e[e] = round_to<T>(f);
    }
    if (wide && n + 4 <= a.N) {
      *reinterpret_cast<u32x2*>(y + n) = v.raw;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < a.N) y[n + e] = v.e[e];
    }
  }
}

template <typename T, int KS>
hipError_t launch_tile_ks(const LinearArgs& a, dim3 grid, hipStream_t st) {
  if (a.glu)
    hipLaunchKernelGGL((linear_tile_kernel<T, true, KS>), grid, dim3(256 * KS), 0, st, a);
  else
    hipLaunchKernelGGL((linear_tile_kernel<T, false, KS>), grid, dim3(256 * KS), 0, st, a);
  return hipGetLastError();
}

// Two groups when every tile of W's rows has a CU to itself: the call is then one
// tile's chain of steps. (All of W's rows, also in the SwiGLU form: its sums are
// then the ones of the product alone.)
template <typename T>
hipError_t launch_tile(const LinearArgs& a, hipStream_t st) {
  const dim3 grid((a.N + kTileRows - 1) / kTileRows, (a.M + kTileRows - 1) / kTileRows);
  const int64_t w_tiles = ((int64_t)a.N * (a.glu ? 2 : 1) + kTileRows - 1) / kTileRows;
  const bool alone = w_tiles * grid.y <= 256 && a.K >= 8 * kTileK;
  return alone ? launch_tile_ks<T, 2>(a, grid, st) : launch_tile_ks<T, 1>(a, grid, st);
}

// 32-bit lane offsets of a tile's loads
bool tile_reaches(const LinearArgs& a) {
  return a.K % kTileK == 0 && (int64_t)a.N * a.K * 2 < (int64_t(1) << 32) &&
         (int64_t)a.M * a.x_st * 2 < (int64_t(1) << 32);
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
  if (a.M > 64 && tile_reaches(a)) return launch_tile<T>(a, st);
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
