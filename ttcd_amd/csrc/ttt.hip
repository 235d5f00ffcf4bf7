// ttt.hip - SwiGLU and the TTT MLP's feature pass for gfx950.
//
// swiglu_kernel replaces fla's swiglu_fwd_kernel (fla/modules/activations.py:
// 412-426, called by swiglu / swiglu_linear in every MLP of the model):
//   z = (g * s) * u,  s = 1 / (1 + exp(-g)),  in fp32, rounded to the dtype.
// Both passes read gate / up with non-temporal loads (each value is used
// once, but for 4 halo rows in 64). Outputs are stored normally: the next op
// reads them soon, from the last-level cache when they fit.
//
// ttt_features_kernel does, in one pass, what the TTT MLP's forward does in
// five launches before its update GEMMs (custom_models/ipttcd/
// modeling_ipttcdv9_lowcopy_scanfuse.py:48-70 with the chunk-local conv of
// profiling/fused_conv.py as patched in by profiling/patches.py:411-432, and
// the group loop's diff at :117-120):
//   z      = swiglu(gate_t, up_t)                teacher features (rounded)
//   zr     = swiglu(gate_s, up_s)                student features (rounded)
//   z_tgt  = conv_t(z), z_hat = conv_s(zr)       chunk-local causal depthwise
//                                                conv, fp32 taps j = 0..K-1,
//                                                each rounded to the dtype
//   diff   = z_tgt - z_hat                       fp32 of the rounded values,
//                                                rounded (chunks 0..T-2 only:
//                                                the last chunk never updates)
// It writes z (the output path reads it), z_hat (the update GEMM reads it)
// and diff; z_tgt and zr never reach HBM. Every intermediate is rounded where
// the reference stores it, so each output equals the reference's chain of
// launches bit for bit (given the same exp).
//
// Layout: rows are tokens, b-major, then chunk, then position in chunk;
// gate / up are the two halves of one (rows, 2*I) GEMM output (row stride
// `gu_stride` elements, gate at column 0, up at column I).
//
// The pass is bound by memory, closely followed by the vector ALU (an exp
// and a reciprocal at quarter rate per value). A lane owns 8 channels (16
// bytes) of a run of 8 positions, and a wavefront 8 such runs one below the
// other: all of a lane's loads are issued before the first is used, a run's
// K-1 halo rows come from the lanes of the run below it, and the halo of the
// wavefront is one extra row, computed by its first K-1 runs side by side.
// Before (one thread per run of 16, a load per row behind the arithmetic of
// the row above, the halo recomputed by every run, expf and a division):
// 24576 rows of 3072 channels, K = 5, 350 us = 3.5 TB/s; now 207 us = 6.0
// TB/s, and 2048 rows of 768 channels 33 -> 15 us. Plain instead of
// non-temporal loads 217 us; three wavefronts per SIMD (spills) 355 us.
//
// The update scan of the group loop (scanfuse.py:121-172) around its GEMMs:
// ttt_pd_beta_t_kernel writes pd * beta (the projected difference scaled by
// the per-token learning rate, :126-127, one bf16 multiply) transposed per
// chunk, (chunk, H, C), so the update GEMM dW_c = pd_c^T z_hat_c (:146-149)
// runs as one batched GEMM on contiguous operands; ttt_scan_kernel then does
// what the reference does in three torch launches per group plus one add per
// chunk (:157-170): the running sum over the group's chunk updates with the
// sum stored in the dtype after every step (torch's GPU scan of a bf16
// tensor), cs_j = lr * sum_j rounded, W_step = W_cur + cs rounded, and the
// next group's W_cur; it writes every chunk's W_step transposed, (step, I, H),
// so the per-chunk output GEMMs z_c W_step^T (:161-165) are one batched GEMM
// on contiguous operands as well. Both transpose through 64 x 64 LDS tiles, in
// 16-byte accesses where the rows allow it (20480 x 1024 pd 39 -> 15 us; 5
// updates of 1024 x 3072 48 -> 16 us) and else by single elements.
// ttt_beta_kernel is the learning rate itself, sigmoid(t . b_proj): one read of
// t (20480 x 1024: 14 us; torch's product and sigmoid 23).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "internal.h"
#include "silu.h"

namespace ttcd {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T>
union V8 {
  u32x4 raw;
  T e[8];
};

template <typename T>
__global__ __launch_bounds__(256) void swiglu_kernel(const T* __restrict__ gate,
                                                     const T* __restrict__ up,
                                                     T* __restrict__ out, int64_t rows, int cols,
                                                     int64_t g_st, int64_t u_st, int64_t o_st) {
  const int ng = cols / 8;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= rows * ng) return;
  const int64_t r = gid / ng;
  const int c = (int)(gid % ng) * 8;
  V8<T> g, u, o;
  g.raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gate + r * g_st + c));
  u.raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(up + r * u_st + c));
#pragma unroll
  for (int e = 0; e < 8; ++e)
    o.e[e] = round_to<T>(silu_mul(static_cast<float>(g.e[e]), static_cast<float>(u.e[e])));
  *reinterpret_cast<u32x4*>(out + r * o_st + c) = o.raw;
}

// Feature pass geometry: a wavefront owns 8 groups of 8 channels (128
// contiguous bytes, lane % 8) of 8 consecutive runs of 8 positions (lane / 8)
// of one chunk.
constexpr int kRunRows = 8;
constexpr int kSegRows = 8 * kRunRows;  // positions per wavefront

// The K taps of 8 neighbouring channels (w + 8 * K elements on): 16-byte loads
// where the weights are aligned to them.
template <typename W, int K>
__device__ __forceinline__ void load_taps(const W* w, bool aligned, float (&wr)[K][8]) {
  constexpr int N = (int)(8 * K * sizeof(W) / 16);
  union {
    u32x4 raw[N];
    W e[8 * K];
  } v;
  if (aligned) {
#pragma unroll
    for (int i = 0; i < N; ++i) v.raw[i] = reinterpret_cast<const u32x4*>(w)[i];
  } else {
#pragma unroll
    for (int i = 0; i < 8 * K; ++i) v.e[i] = w[i];
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int j = 0; j < K; ++j) wr[j][e] = static_cast<float>(v.e[e * K + j]);
}

template <typename T>
__device__ __forceinline__ V8<T> swiglu8(const V8<T>& g, const V8<T>& u) {
  V8<T> f;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    f.e[e] = round_to<T>(silu_mul(static_cast<float>(g.e[e]), static_cast<float>(u.e[e])));
  return f;
}

template <typename T>
__device__ __forceinline__ V8<T> lane_read(const V8<T>& v, int lane) {
  V8<T> r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r.raw[q] = (uint32_t)__shfl((int)v.raw[q], lane, 64);
  return r;
}

// Chunk-local causal conv of a lane's run f, each output rounded. The K-1
// rows before a run are the last ones of the run below it; before the first
// run of the wavefront they are `halo`, row t held by the lanes of run t.
template <typename T, typename W, int K>
__device__ __forceinline__ void conv_run(const V8<T> (&f)[kRunRows], const V8<T>& halo,
                                         const W* w, bool aligned, int lane,
                                         V8<T> (&out)[kRunRows]) {
  static_assert(K - 1 <= kRunRows, "the halo must lie within the previous run");
  float wr[K][8], win[K][8];
  load_taps<W, K>(w, aligned, wr);
#pragma unroll
  for (int t = 0; t < K - 1; ++t) {
    const V8<T> a = lane_read(f[kRunRows - (K - 1) + t], lane - 8);
    const V8<T> h = lane_read(halo, 8 * t + (lane & 7));
#pragma unroll
    for (int e = 0; e < 8; ++e) win[t][e] = static_cast<float>(lane < 8 ? h.e[e] : a.e[e]);
  }
#pragma unroll
  for (int r = 0; r < kRunRows; ++r) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      win[K - 1][e] = static_cast<float>(f[r].e[e]);
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < K; ++j) acc = fmaf(win[j][e], wr[j][e], acc);
      out[r].e[e] = round_to<T>(acc);
    }
#pragma unroll
    for (int t = 0; t < K - 1; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e) win[t][e] = win[t + 1][e];
  }
}

// CT / CS: the teacher / student conv is present (else identity).
template <typename T, typename W, int K, bool CT, bool CS>
__global__ __launch_bounds__(256, 2) void ttt_features_kernel(TttFeatureArgs a, int nseg,
                                                              int ntile, int64_t waves,
                                                              bool w_aligned) {
  const int lane = threadIdx.x & 63;
  const int64_t wid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (wid >= waves) return;  // whole wavefronts leave
  const int tile = (int)(wid % ntile);
  int rest = (int)(wid / ntile);
  const int seg = rest % nseg;
  rest /= nseg;
  const int ch = rest % a.nchunk;
  const int b = rest / a.nchunk;
  const int ng = a.I / 8, dg = tile * 8 + (lane & 7);
  const bool col_ok = dg < ng;
  const int d0 = (col_ok ? dg : ng - 1) * 8;  // idle lanes read a valid group, store nothing
  const int cb = seg * kSegRows;              // first position of the wavefront in its chunk
  const int c0 = cb + (lane >> 3) * kRunRows;
  const int rows = col_ok ? max(0, min(kRunRows, a.C - c0)) : 0;
  const int64_t chunk0 = (int64_t)ch * a.C;
  const int64_t p0 = chunk0 + c0;  // first position of the run in its sequence
  const bool has_diff = ch < a.nchunk - 1;
  const bool has_s = has_diff || a.last_student;

  const T* gt = static_cast<const T*>(a.gu_t) + (int64_t)b * a.t_rows * a.gu_st + d0;
  const T* gs = static_cast<const T*>(a.gu_s) + (int64_t)b * a.s_rows * a.gu_st + d0;
  // Positions past the chunk or the sequence read the last one before (those
  // past the sequence are written as zero, the others not at all).
  const int64_t last = min(a.tokens, chunk0 + a.C) - 1;
  auto at = [&](int64_t p) { return min(p, last) * a.gu_st; };
  // halo row t (chunk position cb - (K-1) + t) by the lanes of run t
  const bool history = K > 1 && cb > 0;
  const int64_t ph = chunk0 + (history ? cb - (K - 1) + min(lane >> 3, K - 2) : 0);

  // every load of the teacher, then of the student, before the first is used
  V8<T> g[kRunRows], u[kRunRows], gh, uh, g2[kRunRows], u2[kRunRows], gh2, uh2;
  auto load = [](const T* p) {
    V8<T> v;
    v.raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return v;
  };
#pragma unroll
  for (int r = 0; r < kRunRows; ++r) {
    g[r] = load(gt + at(p0 + r));
    u[r] = load(gt + at(p0 + r) + a.I);
  }
  if (has_diff && CT && history) {
    gh = load(gt + at(ph));
    uh = load(gt + at(ph) + a.I);
  }
  if (has_s) {
#pragma unroll
    for (int r = 0; r < kRunRows; ++r) {
      g2[r] = load(gs + at(p0 + r));
      u2[r] = load(gs + at(p0 + r) + a.I);
    }
    if (CS && history) {
      gh2 = load(gs + at(ph));
      uh2 = load(gs + at(ph) + a.I);
    }
  }

  V8<T> f[kRunRows], tgt[kRunRows];
  T* z = static_cast<T*>(a.z) + (((int64_t)b * a.nchunk + ch) * a.C + c0) * a.I + d0;
#pragma unroll
  for (int r = 0; r < kRunRows; ++r) {
    f[r] = swiglu8(g[r], u[r]);
    if (p0 + r >= a.tokens) f[r].raw = u32x4{0u, 0u, 0u, 0u};
    if (r < rows) *reinterpret_cast<u32x4*>(z + (int64_t)r * a.I) = f[r].raw;
  }
  if (!has_s) return;
  V8<T> halo;
  if (has_diff) {
    if constexpr (CT) {
      halo.raw = u32x4{0u, 0u, 0u, 0u};
      if (history) halo = swiglu8(gh, uh);
      conv_run<T, W, K>(f, halo, static_cast<const W*>(a.w_t) + (int64_t)d0 * K, w_aligned, lane,
                        tgt);
    } else {
#pragma unroll
      for (int r = 0; r < kRunRows; ++r) tgt[r] = f[r];
    }
  }
#pragma unroll
  for (int r = 0; r < kRunRows; ++r) f[r] = swiglu8(g2[r], u2[r]);
  V8<T> sh[kRunRows];
  if constexpr (CS) {
    halo.raw = u32x4{0u, 0u, 0u, 0u};
    if (history) halo = swiglu8(gh2, uh2);
    conv_run<T, W, K>(f, halo, static_cast<const W*>(a.w_s) + (int64_t)d0 * K, w_aligned, lane,
                      sh);
  } else {
#pragma unroll
    for (int r = 0; r < kRunRows; ++r) sh[r] = f[r];
  }
  const int64_t up_row = ((int64_t)b * (a.nchunk - 1) + ch) * a.C + c0;
  T* zh = static_cast<T*>(a.z_hat) + d0 +
          (a.last_student ? ((int64_t)b * a.nchunk + ch) * a.C + c0 : up_row) * a.I;
  T* df = static_cast<T*>(a.diff) + up_row * a.I + d0;
#pragma unroll
  for (int r = 0; r < kRunRows; ++r) {
    if (r < rows) *reinterpret_cast<u32x4*>(zh + (int64_t)r * a.I) = sh[r].raw;
    if (has_diff) {
      V8<T> d;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        d.e[e] = round_to<T>(static_cast<float>(tgt[r].e[e]) - static_cast<float>(sh[r].e[e]));
      if (r < rows) *reinterpret_cast<u32x4*>(df + (int64_t)r * a.I) = d.raw;
    }
  }
}

template <typename T, typename W, int K, bool CT, bool CS>
hipError_t launch_feat(const TttFeatureArgs& a, hipStream_t st) {
  const int nseg = (a.C + kSegRows - 1) / kSegRows;
  const int ntile = (a.I / 8 + 7) / 8;
  const int64_t waves = (int64_t)a.B * a.nchunk * nseg * ntile;
  const int64_t blocks = (waves + 3) / 4;
  const bool w_aligned = reinterpret_cast<uintptr_t>(a.w_t) % 16 == 0 &&
                         reinterpret_cast<uintptr_t>(a.w_s) % 16 == 0;
  hipLaunchKernelGGL((ttt_features_kernel<T, W, K, CT, CS>), dim3((unsigned)blocks), dim3(256), 0,
                     st, a, nseg, ntile, waves, w_aligned);
  return hipGetLastError();
}

template <typename T, typename W, int K>
hipError_t launch_ck(const TttFeatureArgs& a, hipStream_t st) {
  const bool ct = a.w_t != nullptr, cs = a.w_s != nullptr;
  if (ct && cs) return launch_feat<T, W, K, true, true>(a, st);
  if (ct) return launch_feat<T, W, K, true, false>(a, st);
  if (cs) return launch_feat<T, W, K, false, true>(a, st);
  return launch_feat<T, W, 1, false, false>(a, st);
}

template <typename T, typename W>
hipError_t launch_k(const TttFeatureArgs& a, hipStream_t st) {
  switch (a.K) {
    case 1: return launch_ck<T, W, 1>(a, st);
    case 2: return launch_ck<T, W, 2>(a, st);
    case 3: return launch_ck<T, W, 3>(a, st);
    case 4: return launch_ck<T, W, 4>(a, st);
    case 5: return launch_ck<T, W, 5>(a, st);
    case 6: return launch_ck<T, W, 6>(a, st);
    case 7: return launch_ck<T, W, 7>(a, st);
    default: return launch_ck<T, W, 8>(a, st);
  }
}

template <typename T>
hipError_t launch_wt(const TttFeatureArgs& a, Elem wt, hipStream_t st) {
  switch (wt) {
    case Elem::BF16: return launch_k<T, __bf16>(a, st);
    case Elem::F16: return launch_k<T, _Float16>(a, st);
    default: return launch_k<T, float>(a, st);
  }
}

template <typename T>
hipError_t launch_sw(const void* g, const void* u, void* o, int64_t rows, int cols, int64_t g_st,
                     int64_t u_st, int64_t o_st, hipStream_t st) {
  const int64_t total = rows * (cols / 8);
  const int64_t blocks = (total + 255) / 256;
  hipLaunchKernelGGL(swiglu_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, st,
                     static_cast<const T*>(g), static_cast<const T*>(u), static_cast<T*>(o), rows,
                     cols, g_st, u_st, o_st);
  return hipGetLastError();
}

// 64 x 64 tile transposes for the update scan. Thread (tx, ty) = (tid % 64,
// tid / 64) handles rows ty, ty + 4, ... of a tile; the LDS tile is fp32 with
// a 65-word row pitch, so the transposed reads are free of bank conflicts.
constexpr int kTile = 64;

template <typename T>
__global__ __launch_bounds__(256) void ttt_pd_beta_t_kernel(TttProjBetaArgs a) {
  __shared__ float tile[kTile][kTile + 1];
  const int tx = threadIdx.x % kTile, ty = threadIdx.x / kTile;
  const int h0 = blockIdx.x * kTile, t0 = blockIdx.y * kTile, bk = blockIdx.z;
  const int b = bk / a.nupd, c = bk % a.nupd;
  const T* pd = static_cast<const T*>(a.pd) + (int64_t)bk * a.C * a.pd_stride;
  const T* beta = a.beta ? static_cast<const T*>(a.beta) + b * a.beta_sb + (int64_t)c * a.C
                         : nullptr;
#pragma unroll
  for (int r = 0; r < kTile / 4; ++r) {
    const int t = t0 + ty + 4 * r, h = h0 + tx;
    float v = 0.f;
    if (t < a.C && h < a.H) {
      v = static_cast<float>(pd[(int64_t)t * a.pd_stride + h]);
      // bf16 * bf16 is exact in fp32: one rounding, as the reference's multiply
      if (beta) v = static_cast<float>(round_to<T>(v * static_cast<float>(beta[t])));
    }
    tile[ty + 4 * r][tx] = v;
  }
  __syncthreads();
  T* out = static_cast<T*>(a.pdt) + (int64_t)bk * a.H * a.C;
#pragma unroll
  for (int r = 0; r < kTile / 4; ++r) {
    const int h = h0 + ty + 4 * r, t = t0 + tx;
    if (h < a.H && t < a.C) out[(int64_t)h * a.C + t] = static_cast<T>(tile[tx][ty + 4 * r]);
  }
}

template <typename T>
__device__ __forceinline__ void store_tile_t(float (&tile)[kTile][kTile + 1], const float (&v)[16],
                                             T* out, int h0, int i0, int H, int I, int tx,
                                             int ty) {
  // v[r] is element (h0 + ty + 4r, i0 + tx); out is (I, H): row i, column h
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) tile[ty + 4 * r][tx] = v[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int i = i0 + ty + 4 * r, h = h0 + tx;
    if (i < I && h < H) out[(int64_t)i * H + h] = static_cast<T>(tile[tx][ty + 4 * r]);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void ttt_scan_kernel(TttScanArgs a) {
  __shared__ float tile[kTile][kTile + 1];
  const int tx = threadIdx.x % kTile, ty = threadIdx.x / kTile;
  const int i0 = blockIdx.x * kTile, h0 = blockIdx.y * kTile;
  const int i = i0 + tx;
  const T* wc = static_cast<const T*>(a.w_cur);
  const T* dw = static_cast<const T*>(a.dw);
  T* steps = static_cast<T*>(a.steps_t);
  const int64_t HI = (int64_t)a.H * a.I;
  float w[16], acc[16], ws[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int h = h0 + ty + 4 * r;
    w[r] = (h < a.H && i < a.I) ? static_cast<float>(wc[(int64_t)h * a.I + i]) : 0.f;
    acc[r] = 0.f;
    ws[r] = w[r];
  }
  store_tile_t<T>(tile, w, steps, h0, i0, a.H, a.I, tx, ty);  // step 0: W_cur
  for (int j = 0; j < a.nupd; ++j) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int h = h0 + ty + 4 * r;
      const float d = (h < a.H && i < a.I) ? static_cast<float>(dw[j * HI + (int64_t)h * a.I + i])
                                           : 0.f;
      acc[r] = static_cast<float>(round_to<T>(acc[r] + d));          // running sum, stored
      const float cs = static_cast<float>(round_to<T>(a.lr * acc[r]));  // lr * cumsum
      ws[r] = static_cast<float>(round_to<T>(w[r] + cs));            // W_cur + cs_j
    }
    if (j + 1 < a.nsteps)
      store_tile_t<T>(tile, ws, steps + (int64_t)(j + 1) * HI, h0, i0, a.H, a.I, tx, ty);
  }
  if (a.w_next != nullptr) {
    T* wn = static_cast<T*>(a.w_next);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int h = h0 + ty + 4 * r;
      if (h < a.H && i < a.I) wn[(int64_t)h * a.I + i] = static_cast<T>(ws[r]);
    }
  }
}

// The same two passes on rows of whole 16-byte groups. A thread moves 8
// neighbouring elements of two rows of a 64 x 64 tile at a time; the tile is
// kept transposed in LDS as 16-bit values, at a pitch of 33 words (the 8
// threads of a row then write 8 words apart, and a column is read back as
// words).
constexpr int kTileWords = kTile / 2 + 1;

template <typename T>
struct TileT {
  uint32_t w[kTile * kTileWords];

  // element (row, col + e) of the tile, e = 0..7
  __device__ void put(int row, int col, const V8<T>& v) {
    T* p = reinterpret_cast<T*>(w);
#pragma unroll
    for (int e = 0; e < 8; ++e) p[(col + e) * 2 * kTileWords + row] = v.e[e];
  }
  // elements (row .. row + 7, col)
  __device__ V8<T> get(int row, int col) const {
    V8<T> v;
#pragma unroll
    for (int q = 0; q < 4; ++q) v.raw[q] = w[col * kTileWords + row / 2 + q];
    return v;
  }
};

template <typename T>
__global__ __launch_bounds__(256) void ttt_pd_beta_t_vec_kernel(TttProjBetaArgs a) {
  __shared__ TileT<T> tile;
  const int row = threadIdx.x / 8, col = (threadIdx.x % 8) * 8;
  const int h0 = blockIdx.x * kTile, t0 = blockIdx.y * kTile, bk = blockIdx.z;
  const int b = bk / a.nupd, c = bk % a.nupd;
  const T* pd = static_cast<const T*>(a.pd) + (int64_t)bk * a.C * a.pd_stride;
  const T* beta = a.beta ? static_cast<const T*>(a.beta) + b * a.beta_sb + (int64_t)c * a.C
                         : nullptr;
  V8<T> v[2];
  float be[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int t = min(t0 + row + 32 * r, a.C - 1), h = min(h0 + col, a.H - 8);
    v[r].raw = __builtin_nontemporal_load(
        reinterpret_cast<const u32x4*>(pd + (int64_t)t * a.pd_stride + h));
    be[r] = beta ? static_cast<float>(beta[t]) : 1.f;
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (beta) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[r].e[e] = round_to<T>(static_cast<float>(v[r].e[e]) * be[r]);
    }
    tile.put(row + 32 * r, col, v[r]);
  }
  __syncthreads();
  T* out = static_cast<T*>(a.pdt) + (int64_t)bk * a.H * a.C;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int h = h0 + row + 32 * r, t = t0 + col;
    if (h < a.H && t < a.C)
      *reinterpret_cast<u32x4*>(out + (int64_t)h * a.C + t) = tile.get(col, row + 32 * r).raw;
  }
}

// One step's chunk update is requested while the one before it is folded, and
// two tiles alternate, so a step has one barrier.
template <typename T>
__global__ __launch_bounds__(256) void ttt_scan_vec_kernel(TttScanArgs a) {
  __shared__ TileT<T> tile[2];
  const int row = threadIdx.x / 8, col = (threadIdx.x % 8) * 8;
  const int i0 = blockIdx.x * kTile, h0 = blockIdx.y * kTile;
  const int64_t HI = (int64_t)a.H * a.I;
  int64_t off[2];
  bool ok[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int h = h0 + row + 32 * r, i = i0 + col;
    ok[r] = h < a.H && i < a.I;
    off[r] = (int64_t)min(h, a.H - 1) * a.I + min(i, a.I - 8);
  }
  auto load = [&](const void* p, int64_t at) {
    V8<T> v;
    v.raw = __builtin_nontemporal_load(
        reinterpret_cast<const u32x4*>(static_cast<const T*>(p) + at));
    return v;
  };
  T* steps = static_cast<T*>(a.steps_t);
  auto store_t = [&](const V8<T> (&v)[2], int step) {
    TileT<T>& tl = tile[step & 1];
#pragma unroll
    for (int r = 0; r < 2; ++r) tl.put(row + 32 * r, col, v[r]);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int i = i0 + row + 32 * r, h = h0 + col;
      if (i < a.I && h < a.H)
        *reinterpret_cast<u32x4*>(steps + step * HI + (int64_t)i * a.H + h) =
            tl.get(col, row + 32 * r).raw;
    }
  };
  V8<T> w[2], ws[2], d[2];
  float acc[2][8];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    w[r] = ws[r] = load(a.w_cur, off[r]);
    if (a.nupd > 0) d[r] = load(a.dw, off[r]);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[r][e] = 0.f;
  }
  store_t(w, 0);  // step 0: W_cur
  for (int j = 0; j < a.nupd; ++j) {
    V8<T> nx[2];
#pragma unroll
    for (int r = 0; r < 2; ++r)
      nx[r] = load(a.dw, (j + 1 < a.nupd ? (j + 1) * HI : 0) + off[r]);
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        // the running sum stored, lr * sum, W_cur + cs_j, each rounded
        acc[r][e] =
            static_cast<float>(round_to<T>(acc[r][e] + static_cast<float>(d[r].e[e])));
        const float cs = static_cast<float>(round_to<T>(a.lr * acc[r][e]));
        ws[r].e[e] = round_to<T>(static_cast<float>(w[r].e[e]) + cs);
      }
    if (j + 1 < a.nsteps) store_t(ws, j + 1);
#pragma unroll
    for (int r = 0; r < 2; ++r) d[r] = nx[r];
  }
  if (a.w_next != nullptr) {
    T* wn = static_cast<T*>(a.w_next);
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if (ok[r]) *reinterpret_cast<u32x4*>(wn + off[r]) = ws[r].raw;
  }
}

// beta = sigmoid(t . b_proj) per token: a wavefront takes four rows, so that a
// lane has four row loads in flight for one of the weight.
constexpr int kBetaRows = 4;

template <typename T>
__global__ __launch_bounds__(256) void ttt_beta_kernel(TttBetaArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t r0 = (((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6) * kBetaRows;
  const int64_t total = (int64_t)a.B * a.rows;
  if (r0 >= total) return;  // whole wavefronts leave
  const T* src[kBetaRows];
  float acc[kBetaRows];
#pragma unroll
  for (int r = 0; r < kBetaRows; ++r) {
    const int64_t row = min(r0 + r, total - 1);
    const int64_t b = row / a.rows;
    src[r] = static_cast<const T*>(a.t) + (b * a.t_rows + row - b * a.rows) * a.H;
    acc[r] = 0.f;
  }
  const T* w = static_cast<const T*>(a.w);
  for (int c = 8 * lane; c < a.H; c += 8 * 64) {
    V8<T> wv, v[kBetaRows];
    wv.raw = *reinterpret_cast<const u32x4*>(w + c);
#pragma unroll
    for (int r = 0; r < kBetaRows; ++r) v[r].raw = *reinterpret_cast<const u32x4*>(src[r] + c);
#pragma unroll
    for (int r = 0; r < kBetaRows; ++r)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        acc[r] = fmaf(static_cast<float>(v[r].e[e]), static_cast<float>(wv.e[e]), acc[r]);
  }
  float mine = 0.f;
#pragma unroll
  for (int r = 0; r < kBetaRows; ++r) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) acc[r] += __shfl_xor(acc[r], m, 64);
    mine = lane == r ? acc[r] : mine;
  }
  if (lane < kBetaRows && r0 + lane < total) {
    // the product rounded, then its sigmoid, as the two torch launches round
    const float x = static_cast<float>(round_to<T>(mine));
    static_cast<T*>(a.beta)[r0 + lane] = round_to<T>(1.0f / (1.0f + expf(-x)));
  }
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

template <typename T>
hipError_t launch_pdbt(const TttProjBetaArgs& a, hipStream_t st) {
  const dim3 grid((a.H + kTile - 1) / kTile, (a.C + kTile - 1) / kTile, a.B * a.nupd);
  const bool vec = a.H % 8 == 0 && a.C % 8 == 0 && a.pd_stride % 8 == 0 && aligned16(a.pd) &&
                   aligned16(a.pdt);
  if (vec)
    hipLaunchKernelGGL(ttt_pd_beta_t_vec_kernel<T>, grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(ttt_pd_beta_t_kernel<T>, grid, dim3(256), 0, st, a);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_scan(const TttScanArgs& a, hipStream_t st) {
  const dim3 grid((a.I + kTile - 1) / kTile, (a.H + kTile - 1) / kTile, 1);
  const bool vec = a.H % 8 == 0 && a.I % 8 == 0 && aligned16(a.dw) && aligned16(a.w_cur) &&
                   aligned16(a.steps_t) && aligned16(a.w_next);
  if (vec)
    hipLaunchKernelGGL(ttt_scan_vec_kernel<T>, grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(ttt_scan_kernel<T>, grid, dim3(256), 0, st, a);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_beta(const TttBetaArgs& a, hipStream_t st) {
  const int64_t waves = ((int64_t)a.B * a.rows + kBetaRows - 1) / kBetaRows;
  hipLaunchKernelGGL(ttt_beta_kernel<T>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_swiglu(const void* gate, const void* up, void* out, int64_t rows, int cols,
                         int64_t gate_stride, int64_t up_stride, int64_t out_stride, Elem dtype,
                         hipStream_t stream) {
  return dtype == Elem::BF16
             ? launch_sw<__bf16>(gate, up, out, rows, cols, gate_stride, up_stride, out_stride,
                                 stream)
             : launch_sw<_Float16>(gate, up, out, rows, cols, gate_stride, up_stride, out_stride,
                                   stream);
}

hipError_t launch_ttt_features(const TttFeatureArgs& a, Elem dtype, Elem w_dtype,
                               hipStream_t stream) {
  return dtype == Elem::BF16 ? launch_wt<__bf16>(a, w_dtype, stream)
                             : launch_wt<_Float16>(a, w_dtype, stream);
}

hipError_t launch_ttt_proj_beta_t(const TttProjBetaArgs& a, Elem dtype, hipStream_t stream) {
  return dtype == Elem::BF16 ? launch_pdbt<__bf16>(a, stream) : launch_pdbt<_Float16>(a, stream);
}

hipError_t launch_ttt_beta(const TttBetaArgs& a, Elem dtype, hipStream_t stream) {
  return dtype == Elem::BF16 ? launch_beta<__bf16>(a, stream) : launch_beta<_Float16>(a, stream);
}

hipError_t launch_ttt_scan(const TttScanArgs& a, Elem dtype, hipStream_t stream) {
  return dtype == Elem::BF16 ? launch_scan<__bf16>(a, stream) : launch_scan<_Float16>(a, stream);
}

}  // namespace ttcd
