// fp32 N,C,H,W first layer of the ImageNet networks: 3 -> 64 channels, 7x7,
// stride 2, pad 3, with bias and activation, and optionally the 3x3 stride-2
// pad-1 max pooling that follows it, in one kernel.
//
// At batch 1 the layer is 236 MFLOP over 12544 pixels: what matters is how
// few dependent memory round trips a launch has, not its arithmetic rate.  A
// workgroup owns a tile of 5 rows x 16 columns of convolution pixels and all
// 64 filters.  It reads the tile's input patch (3 x 15 x 37 values, each once,
// zeros outside the image) into LDS, each lane reads its 37 filter values
// into registers at the same time, and after one barrier the whole reduction
// (147 taps, 37 steps of v_mfma_f32_16x16x4_f32) runs out of LDS and
// registers: wavefront w owns filters 16w .. 16w+15, an MFMA column block is
// one row of the tile.  The im2col offset of tap k inside the patch comes
// from a 148-entry table in LDS; tap 147 (the reduction padded to a multiple
// of four) multiplies a zero filter value by a word of a zeroed LDS region,
// so that no non-finite input can leak into the sum through it.
//
// With the pooling: the tile is the 5 x 15 convolution pixels under 2 x 7
// pooled ones (neighbouring tiles recompute the shared row and column: 1.34x
// the arithmetic, no carried state, 224 workgroups at 224 x 224).  A lane
// holds one column of all five rows, so the vertical maxima are in registers
// and the horizontal ones two lane shifts away.  The activation is applied
// after the maximum (both supported ones are monotonic); a NaN anywhere in a
// window gives NaN, as the pooling kernel does.
#include "conv_f32_stem.h"

#include <algorithm>
#include <type_traits>

namespace dnnrt {

namespace stem32 {
constexpr int ROWS = 5, COLS = 16;           // convolution pixels per tile
constexpr int PR = 2 * (ROWS - 1) + 7;       // 15 patch rows
constexpr int PW = 2 * (COLS - 1) + 7;       // 37 patch columns
constexpr int PATCH = 3 * PR * PW;           // values
constexpr int ZEROS = 2 * (COLS - 1) + 2 * PW * (ROWS - 1) + 1;  // words the padding tap can reach
constexpr int TAPS = 147, STEPS = 37;
constexpr int PATCH_LOADS = (PATCH + 255) / 256;
}  // namespace stem32

typedef float floatx4 __attribute__((ext_vector_type(4)));

// The larger of two values, NaN if either is one.
__device__ __forceinline__ float nan_max(float a, float b) {
  const float m = a > b ? a : b;
  return (a != a) ? a : ((b != b) ? b : m);
}

template <bool POOL, bool RELU>
__global__ __launch_bounds__(256) void conv_f32_stem_kernel(const float *__restrict__ X, const float *__restrict__ Wt,
                                                            const float *__restrict__ bias, const float *Zr, float *Y,
                                                            const int H, const int W, const int P, const int Q, const int PP,
                                                            const int QQ, const int tiles_r, const int tiles_c,
                                                            const int w_filter_stride, const int w_tap_stride, const int act,
                                                            const float act_coef) {
  using namespace stem32;
  __shared__ float patch[PATCH + ZEROS];
  __shared__ int tap_offset[4 * STEPS];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, quad = lane >> 4;
  int b = blockIdx.x;
  const int tc = b % tiles_c; b /= tiles_c;
  const int tr = b % tiles_r;
  const int n = b / tiles_r;
  // first convolution pixel of the tile (may be -1 with the pooling: the pooling's own padding)
  const int cr0 = POOL ? 4 * tr - 1 : ROWS * tr, cc0 = POOL ? 14 * tc - 1 : COLS * tc;
  const int ih0 = 2 * cr0 - 3, iw0 = 2 * cc0 - 3;

  // ---- requests: the patch, the lane's filter values, its bias values ----
  const float *xn = X + (int64_t)n * 3 * H * W;
  float pv[PATCH_LOADS];
#pragma unroll
  for (int i = 0; i < PATCH_LOADS; i++) {
    const int e = tid + 256 * i;
    const int c = e / (PR * PW), rem = e - c * (PR * PW), pr = rem / PW, pc = rem - pr * PW;
    const int ih = ih0 + pr, iw = iw0 + pc;
    const bool ok = e < PATCH && (unsigned)ih < (unsigned)H && (unsigned)iw < (unsigned)W;
    const float v = xn[ok ? ((int64_t)c * H + ih) * W + iw : 0];
    pv[i] = ok ? v : 0.f;
  }
  const int filter = 16 * wave + col;
  float a[STEPS];
#pragma unroll
  for (int t = 0; t < STEPS; t++) {
    const int k = 4 * t + quad;
    const float v = Wt[(int64_t)filter * w_filter_stride + (int64_t)(k < TAPS ? k : TAPS - 1) * w_tap_stride];
    a[t] = k < TAPS ? v : 0.f;
  }
  float bv[4];
#pragma unroll
  for (int i = 0; i < 4; i++) bv[i] = bias[16 * wave + 4 * quad + i];

  // ---- LDS: tap table, patch, the zeroed words behind it ----
  if (tid < 4 * STEPS) {
    const int k = tid;
    const int c = (k * 1338) >> 16, rem = k - 49 * c, r = (rem * 9363) >> 16, s = rem - 7 * r;  // k = (c * 7 + r) * 7 + s
    tap_offset[k] = k < TAPS ? (c * PR + r) * PW + s : PATCH;
  }
  for (int e = tid; e < ZEROS; e += 256) patch[PATCH + e] = 0.f;
#pragma unroll
  for (int i = 0; i < PATCH_LOADS; i++) {
    const int e = tid + 256 * i;
    if (e < PATCH) patch[e] = pv[i];
  }
  __syncthreads();

  int off[STEPS];
#pragma unroll
  for (int t = 0; t < STEPS; t++) off[t] = tap_offset[4 * t + quad] + 2 * col;

  floatx4 acc[ROWS];
#pragma unroll
  for (int j = 0; j < ROWS; j++) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < STEPS; t++) {
    float bj[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; j++) bj[j] = patch[off[t] + j * 2 * PW];
#pragma unroll
    for (int j = 0; j < ROWS; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], bj[j], acc[j], 0, 0, 0);
  }

  // acc[j][i]: filter 16 * wave + 4 * quad + i, tile row j, tile column col
  const int f0 = 16 * wave + 4 * quad;
  if constexpr (POOL) {
    const float ninf = -__builtin_inff();
    const bool col_ok = col < 15 && (unsigned)(cc0 + col) < (unsigned)Q;
    const int pr0 = 2 * tr, pc0 = 7 * tc;
    const int q = col >> 1;
    const bool writer = !(col & 1) && q < 7 && pc0 + q < QQ;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float v[ROWS];
#pragma unroll
      for (int j = 0; j < ROWS; j++) v[j] = (col_ok && (unsigned)(cr0 + j) < (unsigned)P) ? acc[j][i] + bv[i] : ninf;
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const float m = nan_max(nan_max(v[2 * p], v[2 * p + 1]), v[2 * p + 2]);
        const float m1 = __shfl_down(m, 1, 16), m2 = __shfl_down(m, 2, 16);
        float h = nan_max(nan_max(m, m1), m2);
        if (RELU) h = h < 0.f ? 0.f : h;
        if (h != h) h = __builtin_nanf("");
        if (writer && pr0 + p < PP) Y[(((int64_t)n * 64 + f0 + i) * PP + pr0 + p) * QQ + pc0 + q] = h;
      }
    }
  } else {
    const bool col_ok = cc0 + col < Q;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < ROWS; j++)
        if (col_ok && cr0 + j < P) {
          const int64_t at = (((int64_t)n * 64 + f0 + i) * P + cr0 + j) * Q + cc0 + col;
          float v = acc[j][i] + bv[i];
          if (Zr) v += Zr[at];  // the residual operand (which may be Y itself: same thread, same element)
          Y[at] = apply_act(v, act, act_coef);
        }
  }
}

// Many tiles (batches): the same layer on workgroups that walk down a column of tiles, four rows of convolution pixels a step.  Filters,
// bias and every index are set up once a walk, the next step's patch is requested before this one's products, and with the
// pooling the row that two steps share is carried in registers instead of computed twice (1.14x the arithmetic instead of
// 1.43x).  An fp32 MFMA and vector instructions take turns on a SIMD, so what each tile did beside its products was a
// third of its time.  224x224 with the pooling, batch 32: a tile a workgroup 132 us, walks 105; batch 64: 223 and 184; without
// it, batch 32: 100.
namespace stem32w {
constexpr int ROWS = 4, COLS = 16, PR = 2 * (ROWS - 1) + 7, PW = 2 * (COLS - 1) + 7, PATCH = 3 * PR * PW;
[[maybe_unused]] constexpr int ZEROS = 2 * (COLS - 1) + 2 * PW * (ROWS - 1) + 1, STAGE = PATCH + ZEROS;
[[maybe_unused]] constexpr int TAPS = stem32::TAPS, STEPS = stem32::STEPS, LOADS = (PATCH + 255) / 256;
}  // namespace stem32w

template <bool POOL, bool RELU>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void conv_f32_stem_walk_kernel(const float *__restrict__ X, const float *__restrict__ Wt,
                                                                 const float *__restrict__ bias, const float *Zr, float *Y,
                                                                 const int H, const int W, const int P, const int Q, const int PP,
                                                                 const int QQ, const int walks, const int steps, const int tiles_c,
                                                                 const int w_filter_stride, const int w_tap_stride, const int act,
                                                                 const float act_coef) {
#if __HIP_DEVICE_COMPILE__
  using namespace stem32w;
  __shared__ float patch[2 * STAGE];
  __shared__ int tap_offset[4 * STEPS];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, quad = lane >> 4;
  int b = blockIdx.x;
  const int tc = b % tiles_c; b /= tiles_c;
  const int walk = b % walks;
  const int n = b / walks;
  // step s has convolution rows 4 s .. 4 s + 3 and, with the pooling, pooled rows 2 s and 2 s + 1; column 0 is the pooling's padding
  const int first = walk * steps, last = min(first + steps, (P + ROWS - 1) / ROWS);
  const int cc0 = POOL ? 14 * tc - 1 : COLS * tc, iw0 = 2 * cc0 - 3;

  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(X) + (int64_t)n * 3 * H * W, 0, 12 * H * W, 0x00020000);
  int row_of[LOADS];      // of the patch; far outside for values in no image column
  unsigned at_of[LOADS];  // byte offset at patch row 0 on image row 0
#pragma unroll
  for (int i = 0; i < LOADS; i++) {
    const int e = tid + 256 * i;
    const int c = e / (PR * PW), rem = e - c * (PR * PW), pr = rem / PW, pc = rem - pr * PW;
    row_of[i] = e < PATCH && (unsigned)(iw0 + pc) < (unsigned)W ? pr : -(1 << 30);
    at_of[i] = 4u * (unsigned)((c * H + pr) * W + iw0 + pc);
  }
  float pv[LOADS];
  auto request = [&](int s) {
    const int ih0 = 2 * ROWS * s - 3;
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
      const unsigned at = (unsigned)(row_of[i] + ih0) < (unsigned)H ? at_of[i] + 4u * (unsigned)(ih0 * W) : 0x80000000u;  // past the end: zero
      pv[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)at, 0, 0));
    }
  };
  const bool carry_in = POOL && first > 0;  // the row above the walk has to be computed for its first step
  request(carry_in ? first - 1 : first);

  const int filter = 16 * wave + col, f0 = 16 * wave + 4 * quad;
  float a[STEPS];
#pragma unroll
  for (int t = 0; t < STEPS; t++) {
    const int k = 4 * t + quad;
    const float v = Wt[(int64_t)filter * w_filter_stride + (int64_t)(k < TAPS ? k : TAPS - 1) * w_tap_stride];
    a[t] = k < TAPS ? v : 0.f;
  }
  float bv[4];
#pragma unroll
  for (int i = 0; i < 4; i++) bv[i] = bias[f0 + i];
  if (tid < 4 * STEPS) {
    const int k = tid;
    const int c = (k * 1338) >> 16, rem = k - 49 * c, r = (rem * 9363) >> 16, s = rem - 7 * r;  // k = (c * 7 + r) * 7 + s
    tap_offset[k] = k < TAPS ? (c * PR + r) * PW + s : PATCH;
  }
  for (int e = tid; e < ZEROS; e += 256) patch[PATCH + e] = patch[STAGE + PATCH + e] = 0.f;
  auto place = [&](float *to) {
#pragma unroll
    for (int i = 0; i < LOADS; i++)
      if (tid + 256 * i < PATCH) to[tid + 256 * i] = pv[i];
  };
  place(patch);
  __syncthreads();
  int off[STEPS];
#pragma unroll
  for (int t = 0; t < STEPS; t++) off[t] = tap_offset[4 * t + quad] + 2 * col;

  const float ninf = -__builtin_inff();
  const bool col_ok = (!POOL || col < 15) && (unsigned)(cc0 + col) < (unsigned)Q;
  float above[4] = {ninf, ninf, ninf, ninf};  // POOL: the convolution row above the step
  auto lds_barrier = []() {  // loads and stores stay in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto step = [&](int s, auto stage_c, bool more) {
    constexpr int STAGE_AT = decltype(stage_c)::value * STAGE, OTHER_AT = STAGE - STAGE_AT;
    if (more) request(s + 1);
    floatx4 acc[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; j++) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < STEPS; t++) {
      float bj[ROWS];
#pragma unroll
      for (int j = 0; j < ROWS; j++) bj[j] = patch[off[t] + STAGE_AT + j * 2 * PW];
#pragma unroll
      for (int j = 0; j < ROWS; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], bj[j], acc[j], 0, 0, 0);
    }
    if (more) place(patch + OTHER_AT);
    // acc[j][i]: filter f0 + i, row 4 s + j, column cc0 + col
    if constexpr (POOL) {
      const int pc0 = 7 * tc, q = col >> 1;
      const bool writer = !(col & 1) && q < 7 && pc0 + q < QQ;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float v[ROWS + 1];
        v[0] = above[i];
#pragma unroll
        for (int j = 0; j < ROWS; j++) v[j + 1] = col_ok && ROWS * s + j < P ? acc[j][i] + bv[i] : ninf;
        above[i] = v[ROWS];
#pragma unroll
        for (int p = 0; p < 2; p++) {
          const float m = nan_max(nan_max(v[2 * p], v[2 * p + 1]), v[2 * p + 2]);
          const float m1 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, m), 0x101, 0xf, 0xf, true));  // the next column's
          const float m2 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, m), 0x102, 0xf, 0xf, true));
          float h = nan_max(nan_max(m, m1), m2);
          if (RELU) h = h < 0.f ? 0.f : h;
          if (h != h) h = __builtin_nanf("");
          if (writer && 2 * s + p < PP) Y[(((int64_t)n * 64 + f0 + i) * PP + 2 * s + p) * QQ + pc0 + q] = h;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < ROWS; j++)
          if (col_ok && ROWS * s + j < P) {
            const int64_t at = (((int64_t)n * 64 + f0 + i) * P + ROWS * s + j) * Q + cc0 + col;
            float v = acc[j][i] + bv[i];
            if (Zr) v += Zr[at];  // the residual operand (which may be Y itself: same thread, same element)
            Y[at] = apply_act(v, act, act_coef);
          }
    }
    lds_barrier();  // every wavefront has read this stage and written its part of the other
  };
  int s = first;
  if (carry_in) {  // the last row of the step above, alone
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    request(first);
#pragma unroll
    for (int t = 0; t < STEPS; t++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], patch[off[t] + (ROWS - 1) * 2 * PW], acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) above[i] = col_ok ? acc[i] + bv[i] : ninf;
    place(patch + STAGE);
    lds_barrier();
    step(s, std::integral_constant<int, 1>{}, s + 1 < last);
    s++;
  }
  for (; s + 1 < last; s += 2) {
    step(s, std::integral_constant<int, 0>{}, true);
    step(s + 1, std::integral_constant<int, 1>{}, s + 2 < last);
  }
  if (s < last) step(s, std::integral_constant<int, 0>{}, false);
#endif
}

bool launch_conv_f32_stem(const dnnrtContext *ctx, int N, int H, int W, int P, int Q, const float *X, const float *Wt,
                          const float *bias, const float *Z, int act, float *Y, bool pool, int PP, int QQ) {
  using namespace stem32;
  if ((int64_t)3 * H * W >= (1ll << 31)) { set_error("first-layer kernel: image too large"); return false; }
  if (!bias) { set_error("first-layer kernel: needs a bias"); return false; }
  if (pool && act != DNNRT_ACT_RELU && act != DNNRT_ACT_IDENTITY) { set_error("conv+maxpool: activation must be ReLU or identity"); return false; }
  if (pool && Z) { set_error("conv+maxpool: no residual operand"); return false; }
  const bool crsk = ctx->filter_layout == DNNRT_FILTER_CRSK;
  const int fs = crsk ? 1 : TAPS, ts = crsk ? 64 : 1;
  const int tiles_r = pool ? (PP + 1) / 2 : (P + ROWS - 1) / ROWS;
  const int tiles_c = pool ? (QQ + 6) / 7 : (Q + COLS - 1) / COLS;
  const int64_t grid = (int64_t)N * tiles_r * tiles_c;
  if (grid > INT32_MAX) { set_error("first-layer kernel: batch too large"); return false; }
  if (grid == 0) return true;
  // Walks of at least four steps on three workgroups per compute unit, which is what the registers hold at a time.
  const int64_t steps_all = ceil_div(P, stem32w::ROWS), columns = (int64_t)N * tiles_c;
  const int steps = (int)ceil_div(steps_all, std::min(steps_all, std::max<int64_t>(1, (int64_t)3 * ctx->num_cu / columns)));
  if (steps >= 4 && columns * steps_all >= 8 * (int64_t)ctx->num_cu && (int64_t)12 * H * W < (1ll << 31)) {
    const int walks = (int)ceil_div(steps_all, steps);
#define STEM32W(POOL, RELU)                                                                                                                   \
  hipLaunchKernelGGL((conv_f32_stem_walk_kernel<POOL, RELU>), dim3((unsigned)((int64_t)N * walks * tiles_c)), dim3(256), 0, ctx->stream, X, Wt, \
                     bias, Z, Y, H, W, P, Q, PP, QQ, walks, steps, tiles_c, fs, ts, act, ctx->act_coef)
    if (!pool) STEM32W(false, false);
    else if (act == DNNRT_ACT_RELU) STEM32W(true, true);
    else STEM32W(true, false);
#undef STEM32W
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { set_error("first-layer kernel: launch failed: %s", hipGetErrorString(e)); return false; }
    return true;
  }
#define STEM32(POOL, RELU)                                                                                                  \
  hipLaunchKernelGGL((conv_f32_stem_kernel<POOL, RELU>), dim3((unsigned)grid), dim3(256), 0, ctx->stream, X, Wt, bias, Z, Y, H,     \
                     W, P, Q, PP, QQ, tiles_r, tiles_c, fs, ts, act, ctx->act_coef)
  if (pool) {
    if (act == DNNRT_ACT_RELU) STEM32(true, true);
    else STEM32(true, false);
  } else {
    STEM32(false, false);
  }
#undef STEM32
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("first-layer kernel: launch failed: %s", hipGetErrorString(e)); return false; }
  return true;
}

}  // namespace dnnrt
