// silu.h - the SwiGLU arithmetic shared by ttt.hip and linear.hip, so that
// every kernel that forms a SwiGLU value rounds it the same.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

namespace ttcd {
namespace {

// Rounded to T as a separate step from the fp32 result (no fused
// multiply-and-convert), as the reference stores an fp32 value.
template <typename T>
__device__ __forceinline__ T round_to(float v) {
  asm volatile("" : "+v"(v));
  return static_cast<T>(v);
}

// (g * s) * u with s = 1 / (1 + exp(-g)) in fp32. exp(-g) = 2^hi (1 + lo ln 2)
// with hi + lo = -g log2(e) to ~48 bits, and one Newton step on the
// reciprocal: 14 VALU operations beside the two quarter-rate ones, where expf
// and the division take 25 and more. The denominator is held as d / 16: up to
// the largest finite one its reciprocal is then normal (the instruction
// flushes subnormal results), and s itself is the subnormal that a division
// gives. Past |g| = 120 the exponential is 0 or infinite either way; an
// infinite denominator keeps its reciprocal 0.
__device__ __forceinline__ float silu_mul(float g, float u) {
  constexpr float kLog2e = 1.44269504088896341f;
  constexpr float kLog2eLo = (float)(1.44269504088896340736 - (double)kLog2e);
  constexpr float kLn2 = 0.693147180559945309f;
  constexpr float kScale = 0.0625f;
  const float n = __builtin_amdgcn_fmed3f(-g, -120.f, 120.f);
  const float hi = n * kLog2e;
  const float lo = fmaf(n, kLog2eLo, fmaf(n, kLog2e, -hi));
  const float d =
      fmaf(__builtin_amdgcn_exp2f(hi), fmaf(lo, kLn2 * kScale, kScale), kScale);  // d / 16
  const float r = __builtin_amdgcn_rcpf(d);
  const float s = (d < INFINITY ? fmaf(fmaf(-d, r, 1.0f), r, r) : r) * kScale;
  return (g * s) * u;
}

}  // namespace
}  // namespace ttcd
