// Shared declarations of the gfx950 runtime library: the handle, error
// reporting and small host helpers.  Everything here is internal; the public
// surface is include/dnnrt.h.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/dnnrt.h"
#include "lds_limit.h"

// A cut of an inverted residual block (conv_f16_block.hip, conv_f32_block.hip) and the sizes it was found for.
struct dnnrtBlockCut {
  int64_t sizes[11];
  int nb, qw, waves, splits;
};

struct dnnrtContext {
  hipStream_t stream;  // kernels of this handle are launched here
  int format;          // DNNRT_NCHW / DNNRT_NHWC / DNNRT_NCHW_TO_NHWC
  int filter_layout;   // DNNRT_FILTER_KCRS / DNNRT_FILTER_CRSK (fp32 convolutions)
  float act_coef;      // ceiling of CLIPPED_RELU / slope of LEAKY_RELU
  int device;
  int num_cu;
  // Scratch for reductions split over workgroups: partial tiles and one
  // arrival counter per output tile (all zero between kernels).  The library's
  // static array for the first live handle of a device, allocated for any
  // further one; kernels of one handle run in stream order, so they share it.
  float *splitk_partials;
  unsigned *splitk_counters;
  int64_t splitk_partial_bytes;  // what the two buffers hold
  int splitk_max_tiles;
  // The buffers are shared with callers this handle knows nothing of (the process-wide static scratch of
  // dnnrtConvBiasActivNoAlloc): clear the counters a launch uses before it, and refuse a problem whose
  // split would have to shrink to fit instead of shrinking it.
  bool splitk_shared;
  bool scratch_is_static;  // the two buffers are the library's static array (held by one handle per device), not allocations
  // The cuts found last, a ring: a search takes 20 to 60 us, as long as several launches.  A handle is used by one thread at a time.
  mutable dnnrtBlockCut block_cuts[32];
  mutable unsigned block_cuts_found;
  int f16_tile;        // dnnrtSetConvTile: 0 = pick the fp16 convolution variant by problem size, otherwise one of F16_TILE_IDS
};

namespace dnnrt {

constexpr int64_t SPLITK_PARTIAL_BYTES = 8ll << 20;  // a handle's scratch: 2048 partial 32x32 fp32 tiles
constexpr int SPLITK_MAX_TILES = 16384;               // ... and arrival counters
// The static scratch of dnnrtConvBiasActivNoAlloc (conv.hip): the split-reduction convolution kernels ask for
// at most one partial tile per compute unit, 1 MiB on 256 of them.
constexpr int64_t NOALLOC_PARTIAL_BYTES = 1ll << 20;
constexpr int NOALLOC_MAX_TILES = 1024;

// The fp16 channels-last convolution variants dnnrtSetConvTile can force
// (zero-terminated; what each one is: launch_conv_f16 in conv_f16.hip).
constexpr int F16_TILE_IDS[] = {3, 4, 11, 12, 15, 17, 18, 31, 32, 33, 34, 35, 36, 37, 38, 39, 40, 60, 61, 62, 63, 64, 65, 66, 67, 69,
                                  41, 42, 43, 44, 45, 46, 47, 48, 49, 51, 52, 54, 57, 70, 0};

void set_error(const char *fmt, ...) __attribute__((format(printf, 1, 2)));

// Compute entry points return NULL on error.
#define DNNRT_FAIL(...)                                                        \
  do {                                                                         \
    ::dnnrt::set_error(__VA_ARGS__);                                           \
    return nullptr;                                                            \
  } while (0)

#define DNNRT_CHECK_LAUNCH(what)                                               \
  do {                                                                         \
    hipError_t e_ = hipGetLastError();                                         \
    if (e_ != hipSuccess) DNNRT_FAIL("%s: launch failed: %s", what, hipGetErrorString(e_)); \
  } while (0)

inline int64_t numel(const int64_t *d, int64_t rank) {
  int64_t n = 1;
  for (int64_t i = 0; i < rank; i++) n *= d[i];
  return n;
}
inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline bool float_dtype(int32_t dt) { return dt == DNNRT_F32 || dt == DNNRT_F16; }

// Gelu as an epilogue of the matrix products only (not an activMode of the convolution calls).
constexpr int ACT_GELU = 7;

// The activations a convolution epilogue can apply (sigmoid and tanh are
// separate calls, as in the reference).
// x / d for 0 <= x < 2^31 with magic = magic_of(d) from the host: one
// multiply-high and a correction instead of ~40 instructions of integer division.
__device__ __forceinline__ int div_magic(int x, int d, unsigned magic) {
  int q = (int)__umulhi((unsigned)x, magic);
  int r = x - q * d;
  if (r < 0) { q--; r += d; }
  if (r >= d) q++;
  return q;
}
inline unsigned magic_of(int d) {  // ceil(2^32 / d), saturated (d == 1)
  const uint64_t m = (((uint64_t)1 << 32) + (uint64_t)d - 1) / (uint64_t)d;
  return (unsigned)(m > 0xffffffffull ? 0xffffffffull : m);
}

// v / 2 (1 + erf(v / sqrt 2)) without a branch: erff's two ranges, both taken by some lane of nearly every wavefront, made an
// epilogue of sixteen values 2.2 us long.  |v| >= 1: erfc(a) = t P(t) exp(-a^2), t = 1 / (1 + 0.44 a) (the form of Abramowitz
// and Stegun 7.1.26), below: erf(v / sqrt 2) = v R(v^2); P and R are minimax fits (2.2e-9 and 2.6e-10 absolute).  Relative error
// in the 2-norm against 64 bits over normal v of deviation 0.1, 0.5, 1, 4: 3.7e-8, 4.0e-8, 3.5e-8, 2.1e-8; by way of erff
// 3.8e-8, 4.2e-8, 3.9e-8, 2.3e-8.
__device__ __forceinline__ float gelu(float v) {
  const float a = fabsf(v) * 0.70710678118654752f, t = __builtin_amdgcn_rcpf(fmaf(0.44f, a, 1.0f)), u = v * v;
  float p = 0.09016146510839462f;
  p = fmaf(p, t, -0.5130200386047363f);
  p = fmaf(p, t, 0.9627975821495056f);
  p = fmaf(p, t, -0.4957951605319977f);
  p = fmaf(p, t, 0.5246581435203552f);
  p = fmaf(p, t, 0.17550785839557648f);
  p = fmaf(p, t, 0.2556901276111603f) * t;
  float r = -1.506052831246052e-05f;
  r = fmaf(r, u, 0.0002262870839331299f);
  r = fmaf(r, u, -0.0023719691671431065f);
  r = fmaf(r, u, 0.019946342334151268f);
  r = fmaf(r, u, -0.13298065960407257f);
  r = fmaf(r, u, 0.7978845834732056f);
  const float e = __builtin_amdgcn_exp2f(a * (a * -1.4426950408889634f));
  const float outer = v < 0.f ? p * e : fmaf(-p, e, 2.0f);
  return (0.5f * v) * (a < 0.70710678f ? fmaf(v, r, 1.0f) : outer);
}
__device__ __forceinline__ float apply_act(float v, int act, float coef) {
  if (act == DNNRT_ACT_RELU) return v < 0.f ? 0.f : v;
  if (act == DNNRT_ACT_CLIPPED_RELU) { v = v < 0.f ? 0.f : v; return v > coef ? coef : v; }
  if (act == DNNRT_ACT_LEAKY_RELU) return v < 0.f ? coef * v : v;
  if (act == ACT_GELU) return gelu(v);
  return v;
}
__host__ __device__ inline bool fusable_act(int64_t act) {
  return act == DNNRT_ACT_RELU || act == DNNRT_ACT_IDENTITY || act == DNNRT_ACT_CLIPPED_RELU || act == DNNRT_ACT_LEAKY_RELU;
}

}  // namespace dnnrt
