// Reductions and normalisations: dnnrtReduce (mean), dnnrtSoftmax,
// dnnrtLayerNorm.  Wavefront-per-row kernels: a 64-lane wave walks one row
// with coalesced loads and combines with cross-lane shuffles; no LDS, no
// atomics.  Reference wrappers replaced:
// src/Tools/dnn-wrapper/cudnn/CUDNNReduceFunc.cpp:8-142 and
// src/Tools/dnn-wrapper/cuda/CUDASoftmaxFunc.cu:7-128.
#include "common.h"

#include <type_traits>

namespace dnnrt {

__device__ __forceinline__ float ld_f(const float *p) { return *p; }
__device__ __forceinline__ float ld_f(const __half *p) { return __half2float(*p); }
__device__ __forceinline__ void st_f(float *p, float v) { *p = v; }
__device__ __forceinline__ void st_f(__half *p, float v) { *p = __float2half_rn(v); }

// A value combined over the wavefront, in every lane: DPP within the sixteen lanes of a row, then the rows by swaps.  These are
// vector instructions; six shuffles through the LDS crossbar were 0.2 us a sum, two in a row of a layer normalisation.
template <typename F>
__device__ __forceinline__ float wave_combine(float v, F f) {
#if __HIP_DEVICE_COMPILE__
  auto dpp = [&](auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  v = f(v, dpp(std::integral_constant<int, 0xB1>{}));   // the pair's other lane
  v = f(v, dpp(std::integral_constant<int, 0x4E>{}));   // the quad's other pair
  v = f(v, dpp(std::integral_constant<int, 0x141>{}));  // mirrored within eight: the other quad
  v = f(v, dpp(std::integral_constant<int, 0x140>{}));  // mirrored within sixteen: the other eight
  const auto rows = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  v = f(__builtin_bit_cast(float, (unsigned)rows[0]), __builtin_bit_cast(float, (unsigned)rows[1]));
  const auto halves = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  v = f(__builtin_bit_cast(float, (unsigned)halves[0]), __builtin_bit_cast(float, (unsigned)halves[1]));
#endif
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
  return wave_combine(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_combine(v, [](float a, float b) { return fmaxf(a, b); });
}

// mean over the last (contiguous) L elements of each row
template <typename T>
__global__ __launch_bounds__(256) void mean_rows_kernel(const T *__restrict__ x, T *__restrict__ y,
                                                        int64_t rows, int L) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T *xr = x + row * L;
  float s = 0.f;
  for (int i = lane; i < L; i += 64) s += ld_f(xr + i);
  s = wave_sum(s);
  if (lane == 0) st_f(y + row, s / (float)L);
}

// mean over the middle dim of [outer, red, inner]; one thread per (outer, inner)
template <typename T>
__global__ __launch_bounds__(256) void mean_cols_kernel(const T *__restrict__ x, T *__restrict__ y,
                                                        int64_t outer, int red, int64_t inner) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= outer * inner) return;
  const int64_t o = i / inner, in = i - o * inner;
  const T *xp = x + o * red * inner + in;
  float s = 0.f;
  for (int r = 0; r < red; r++) s += ld_f(xp + (int64_t)r * inner);
  st_f(y + i, s / (float)red);
}

// The same with V consecutive inner elements (8 bytes) per thread and the
// loads of seven reduction steps in flight at a time; the sums run in the
// same order as above.  A channels-last global average pool is this shape
// (49 steps over 2048 channels): with one 2-byte load in flight per lane it
// ran at a tenth of the memory rate.
template <typename T, int V>
__global__ __launch_bounds__(256) void mean_cols_vec_kernel(const T *__restrict__ x, T *__restrict__ y,
                                                            int64_t outer, int red, int64_t inner_v) {
  struct alignas(sizeof(T) * V) Vec { T v[V]; };
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= outer * inner_v) return;
  const int64_t o = i / inner_v, in = i - o * inner_v;
  const Vec *xp = reinterpret_cast<const Vec *>(x) + o * red * inner_v + in;
  float s[V];
#pragma unroll
  for (int e = 0; e < V; e++) s[e] = 0.f;
  int r = 0;
  for (; r + 7 <= red; r += 7) {
    Vec t[7];
#pragma unroll
    for (int u = 0; u < 7; u++) t[u] = xp[(int64_t)(r + u) * inner_v];
#pragma unroll
    for (int u = 0; u < 7; u++)
#pragma unroll
      for (int e = 0; e < V; e++) s[e] += ld_f(&t[u].v[e]);
  }
  for (; r < red; r++) {
    const Vec t = xp[(int64_t)r * inner_v];
#pragma unroll
    for (int e = 0; e < V; e++) s[e] += ld_f(&t.v[e]);
  }
  Vec out;
#pragma unroll
  for (int e = 0; e < V; e++) st_f(&out.v[e], s[e] / (float)red);
  reinterpret_cast<Vec *>(y)[i] = out;
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_rows_kernel(const T *__restrict__ x, T *__restrict__ y,
                                                           int64_t rows, int L) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T *xr = x + row * L;
  T *yr = y + row * L;
  float m = -INFINITY;
  for (int i = lane; i < L; i += 64) m = fmaxf(m, ld_f(xr + i));
  m = wave_max(m);
  float s = 0.f;
  for (int i = lane; i < L; i += 64) s += expf(ld_f(xr + i) - m);
  s = wave_sum(s);
  for (int i = lane; i < L; i += 64) st_f(yr + i, expf(ld_f(xr + i) - m) / s);
}

// softmax over the middle dim of [outer, L, inner], inner > 1
template <typename T>
__global__ __launch_bounds__(256) void softmax_cols_kernel(const T *__restrict__ x, T *__restrict__ y,
                                                           int64_t outer, int L, int64_t inner) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= outer * inner) return;
  const int64_t o = i / inner, in = i - o * inner;
  const T *xp = x + o * L * inner + in;
  T *yp = y + o * L * inner + in;
  float m = -INFINITY;
  for (int l = 0; l < L; l++) m = fmaxf(m, ld_f(xp + (int64_t)l * inner));
  float s = 0.f;
  for (int l = 0; l < L; l++) s += expf(ld_f(xp + (int64_t)l * inner) - m);
  for (int l = 0; l < L; l++) st_f(yp + (int64_t)l * inner, expf(ld_f(xp + (int64_t)l * inner) - m) / s);
}

template <typename T>
__global__ __launch_bounds__(256) void layernorm_kernel(const T *__restrict__ x, const T *__restrict__ g,
                                                        const T *__restrict__ b, T *__restrict__ y,
                                                        int64_t rows, int L, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T *xr = x + row * L;
  T *yr = y + row * L;
  float s = 0.f;
  for (int i = lane; i < L; i += 64) s += ld_f(xr + i);
  const float mu = wave_sum(s) / (float)L;
  float v = 0.f;
  for (int i = lane; i < L; i += 64) { const float d = ld_f(xr + i) - mu; v += d * d; }
  const float inv = 1.0f / sqrtf(wave_sum(v) / (float)L + eps);
  for (int i = lane; i < L; i += 64)
    st_f(yr + i, (ld_f(xr + i) - mu) * inv * ld_f(g + i) + ld_f(b + i));
}

// The same for rows of up to 64 * 4 * V elements (L % 4 == 0): a lane keeps
// its V groups of four in registers, so the row, gamma and beta are read once
// and all of it is requested before anything is waited for.  WAVES rows per
// workgroup: 1 when there are few rows, so that they spread over the CUs.
__device__ __forceinline__ float as_f(float v) { return v; }
__device__ __forceinline__ float as_f(__half v) { return __half2float(v); }
template <typename T> __device__ __forceinline__ T as_t(float v);
template <> __device__ __forceinline__ float as_t<float>(float v) { return v; }
template <> __device__ __forceinline__ __half as_t<__half>(float v) { return __float2half_rn(v); }
template <typename T> struct Vec4;
template <> struct Vec4<float> { typedef float4 type; };
template <> struct Vec4<__half> { struct alignas(8) type { __half x, y, z, w; }; };
template <typename T, int V, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void layernorm_reg_kernel(const T *__restrict__ x, const T *__restrict__ g,
                                                                   const T *__restrict__ b, T *__restrict__ y,
                                                                   int64_t rows, int L, float eps) {
  typedef typename Vec4<T>::type V4;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * WAVES + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int n4 = L >> 2;
  const V4 *xr = reinterpret_cast<const V4 *>(x + row * L);
  const V4 *g4 = reinterpret_cast<const V4 *>(g), *b4 = reinterpret_cast<const V4 *>(b);
  V4 xv[V], gv[V], bv[V];
#pragma unroll
  for (int v = 0; v < V; v++) {
    const int j = min(v * 64 + lane, n4 - 1);  // clamped: the duplicates are left out of the sums below
    xv[v] = xr[j]; gv[v] = g4[j]; bv[v] = b4[j];
  }
  __builtin_amdgcn_sched_barrier(0);  // or the compiler moves some of the loads behind the sums that do not need them
  float f[V][4];
  float s = 0.f;
#pragma unroll
  for (int v = 0; v < V; v++) {
    f[v][0] = as_f(xv[v].x); f[v][1] = as_f(xv[v].y); f[v][2] = as_f(xv[v].z); f[v][3] = as_f(xv[v].w);
    if (v * 64 + lane < n4) s += (f[v][0] + f[v][1]) + (f[v][2] + f[v][3]);
  }
  const float mu = wave_sum(s) / (float)L;
  float q = 0.f;
#pragma unroll
  for (int v = 0; v < V; v++) {
#pragma unroll
    for (int e = 0; e < 4; e++) f[v][e] -= mu;
    if (v * 64 + lane < n4) q += (f[v][0] * f[v][0] + f[v][1] * f[v][1]) + (f[v][2] * f[v][2] + f[v][3] * f[v][3]);
  }
  const float inv = 1.0f / sqrtf(wave_sum(q) / (float)L + eps);
  V4 *yr = reinterpret_cast<V4 *>(y + row * L);
#pragma unroll
  for (int v = 0; v < V; v++) {
    const int j = v * 64 + lane;
    if (j >= n4) continue;
    V4 o;
    o.x = as_t<T>(f[v][0] * inv * as_f(gv[v].x) + as_f(bv[v].x));
    o.y = as_t<T>(f[v][1] * inv * as_f(gv[v].y) + as_f(bv[v].y));
    o.z = as_t<T>(f[v][2] * inv * as_f(gv[v].z) + as_f(bv[v].z));
    o.w = as_t<T>(f[v][3] * inv * as_f(gv[v].w) + as_f(bv[v].w));
    yr[j] = o;
  }
}

// ... and for few rows, where the chain of one row is what the launch takes: W wavefronts on a row, a group of four to a lane, the
// wavefronts' sums through LDS.  In a BERT-base the fp32 rows of 768 (128 tokens, 25 launches) take 642 -> 634 us of the whole, the fp16 ones
// (384 tokens) 527.1 -> 524.7; back to back, 128 rows of 768 2.85 -> 2.77, of 2048 3.29 -> 2.90.
template <typename T, int W>
__global__ __launch_bounds__(64 * W) void layernorm_row_kernel(const T *__restrict__ x, const T *__restrict__ g, const T *__restrict__ b, T *__restrict__ y,
                                                               int L, float eps) {
  typedef typename Vec4<T>::type V4;
  __shared__ float part[2][W];
  const int i = threadIdx.x, n4 = L >> 2, j = min(i, n4 - 1);
  const int64_t first = (int64_t)blockIdx.x * n4;
  const V4 xv = reinterpret_cast<const V4 *>(x)[first + j], gv = reinterpret_cast<const V4 *>(g)[j], bv = reinterpret_cast<const V4 *>(b)[j];
  __builtin_amdgcn_sched_barrier(0);
  auto over_row = [&](float v, int which) {
    v = wave_sum(i < n4 ? v : 0.f);
    if constexpr (W > 1) {
      if ((i & 63) == 0) part[which][i >> 6] = v;
      __syncthreads();
      v = part[which][0];
#pragma unroll
      for (int w = 1; w < W; w++) v += part[which][w];
    }
    return v;
  };
  float f[4] = {as_f(xv.x), as_f(xv.y), as_f(xv.z), as_f(xv.w)};
  const float mu = over_row((f[0] + f[1]) + (f[2] + f[3]), 0) / (float)L;
#pragma unroll
  for (int e = 0; e < 4; e++) f[e] -= mu;
  const float inv = 1.0f / sqrtf(over_row((f[0] * f[0] + f[1] * f[1]) + (f[2] * f[2] + f[3] * f[3]), 1) / (float)L + eps);
  if (i >= n4) return;
  V4 o;
  o.x = as_t<T>(f[0] * inv * as_f(gv.x) + as_f(bv.x));
  o.y = as_t<T>(f[1] * inv * as_f(gv.y) + as_f(bv.y));
  o.z = as_t<T>(f[2] * inv * as_f(gv.z) + as_f(bv.z));
  o.w = as_t<T>(f[3] * inv * as_f(gv.w) + as_f(bv.w));
  reinterpret_cast<V4 *>(y)[first + i] = o;
}

template <typename T, int V>
static void launch_layernorm_reg(const dnnrtContext *ctx, const void *X, const void *g, const void *b, void *Y,
                                 int64_t rows, int L, float eps) {
  // up to twelve wavefronts a compute unit; beyond, what a row takes in all counts (700 fp16 rows of 2048: 3.95 us with eight, 3.76 with one)
  if (rows <= 4 * (int64_t)ctx->num_cu && rows * V <= 12 * (int64_t)ctx->num_cu)
    hipLaunchKernelGGL((layernorm_row_kernel<T, V>), dim3((unsigned)rows), dim3(64 * V), 0, ctx->stream, (const T *)X,
                       (const T *)g, (const T *)b, (T *)Y, L, eps);
  else if (rows <= 4 * (int64_t)ctx->num_cu)
    hipLaunchKernelGGL((layernorm_reg_kernel<T, V, 1>), dim3((unsigned)rows), dim3(64), 0, ctx->stream, (const T *)X,
                       (const T *)g, (const T *)b, (T *)Y, rows, L, eps);
  else
    hipLaunchKernelGGL((layernorm_reg_kernel<T, V, 4>), dim3((unsigned)ceil_div(rows, 4)), dim3(256), 0, ctx->stream,
                       (const T *)X, (const T *)g, (const T *)b, (T *)Y, rows, L, eps);
}
template <typename T>
static bool layernorm_in_registers(const dnnrtContext *ctx, const void *X, const void *g, const void *b, void *Y,
                                   int64_t rows, int64_t L, float eps) {
  const uintptr_t align = 4 * sizeof(T) - 1;
  if (L % 4 || L > 2048 || ((uintptr_t)X & align) || ((uintptr_t)Y & align) || ((uintptr_t)g & align) || ((uintptr_t)b & align))
    return false;
  switch ((int)ceil_div(L, 256)) {
    case 1: launch_layernorm_reg<T, 1>(ctx, X, g, b, Y, rows, (int)L, eps); break;
    case 2: launch_layernorm_reg<T, 2>(ctx, X, g, b, Y, rows, (int)L, eps); break;
    case 3: launch_layernorm_reg<T, 3>(ctx, X, g, b, Y, rows, (int)L, eps); break;
    case 4: launch_layernorm_reg<T, 4>(ctx, X, g, b, Y, rows, (int)L, eps); break;
    case 5: case 6: launch_layernorm_reg<T, 6>(ctx, X, g, b, Y, rows, (int)L, eps); break;
    default: launch_layernorm_reg<T, 8>(ctx, X, g, b, Y, rows, (int)L, eps); break;
  }
  return true;
}

template <typename T>
static bool run_reduce(const dnnrtContext *ctx, const void *X, void *Y, int64_t outer, int64_t red,
                       int64_t inner) {
  if (red > INT32_MAX) { set_error("reduce: reduced extent too large"); return false; }
  if (inner == 1) {
    const int64_t blocks = ceil_div(outer, 4);
    if (blocks > INT32_MAX) { set_error("reduce: too many rows"); return false; }
    hipLaunchKernelGGL((mean_rows_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, ctx->stream,
                       (const T *)X, (T *)Y, outer, (int)red);
  } else {
    constexpr int V = 8 / (int)sizeof(T);
    const bool vec = inner % V == 0 && (reinterpret_cast<uintptr_t>(X) & 7u) == 0 && (reinterpret_cast<uintptr_t>(Y) & 7u) == 0;
    const int64_t blocks = ceil_div(vec ? outer * (inner / V) : outer * inner, 256);
    if (blocks > INT32_MAX) { set_error("reduce: tensor too large"); return false; }
    if (vec)
      hipLaunchKernelGGL((mean_cols_vec_kernel<T, V>), dim3((unsigned)blocks), dim3(256), 0, ctx->stream,
                         (const T *)X, (T *)Y, outer, (int)red, inner / V);
    else
      hipLaunchKernelGGL((mean_cols_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, ctx->stream,
                         (const T *)X, (T *)Y, outer, (int)red, inner);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("reduce: launch failed: %s", hipGetErrorString(e)); return false; }
  return true;
}

}  // namespace dnnrt

using namespace dnnrt;

extern "C" {

void *dnnrtReduce(dnnrtHandle_t handle, int32_t rank, const void *X, const int64_t *dimX, void *Y,
                  const int64_t *dimY, int32_t mode, int32_t dtype) {
  if (!handle) DNNRT_FAIL("dnnrtReduce: null handle");
  if (!X || !Y || !dimX || !dimY) DNNRT_FAIL("dnnrtReduce: null argument");
  if (mode != DNNRT_REDUCE_AVG) DNNRT_FAIL("dnnrtReduce: mode %d (only 5 = AVG)", mode);
  if (rank < 1 || rank > 8) DNNRT_FAIL("dnnrtReduce: rank %d", rank);
  int64_t dx[8], dy[8];
  for (int i = 0; i < rank; i++) { dx[i] = dimX[i]; dy[i] = dimY[i]; }
  for (int i = 0; i < rank; i++)
    if (dimX[i] < 0 || dimY[i] < 0) DNNRT_FAIL("dnnrtReduce: negative dim");
  // an empty batch is no work: nothing is launched and Y is left as it is (the reference's zero-block launches do nothing either)
  if (numel(dimX, rank) == 0 || numel(dimY, rank) == 0) return Y;
  if (handle->format != DNNRT_NCHW && rank == 4) {  // channels-last: dense [N,H,W,C]
    dx[1] = dimX[2]; dx[2] = dimX[3]; dx[3] = dimX[1];
    dy[1] = dimY[2]; dy[2] = dimY[3]; dy[3] = dimY[1];
  }
  // reduced dims must form one contiguous run: [outer, red, inner]
  int64_t outer = 1, red = 1, inner = 1;
  int state = 0;  // 0 before the run, 1 inside, 2 after
  for (int i = 0; i < rank; i++) {
    if (dx[i] <= 0) DNNRT_FAIL("dnnrtReduce: non-positive dim");
    if (dy[i] != dx[i] && dy[i] != 1) DNNRT_FAIL("dnnrtReduce: dimY[%d] must be dimX[%d] or 1", i, i);
    const bool r = dy[i] == 1 && dx[i] != 1;
    if (dx[i] == 1) continue;
    if (r) {
      if (state == 2) DNNRT_FAIL("dnnrtReduce: reduced dims must be adjacent");
      state = 1; red *= dx[i];
    } else {
      if (state == 0) outer *= dx[i];
      else { state = 2; inner *= dx[i]; }
    }
  }
  bool ok;
  if (dtype == DNNRT_F32) ok = run_reduce<float>(handle, X, Y, outer, red, inner);
  else if (dtype == DNNRT_F16) ok = run_reduce<__half>(handle, X, Y, outer, red, inner);
  else DNNRT_FAIL("dnnrtReduce: dtype %d", dtype);
  return ok ? Y : nullptr;
}

void *dnnrtSoftmax(dnnrtHandle_t handle, const void *X, const int64_t *dimX, void *Y,
                   const int64_t *dimY, int64_t axis, int64_t rank, int32_t dtype) {
  (void)dimY;
  if (!handle) DNNRT_FAIL("dnnrtSoftmax: null handle");
  if (!X || !Y || !dimX) DNNRT_FAIL("dnnrtSoftmax: null argument");
  if (rank < 1 || rank > 8) DNNRT_FAIL("dnnrtSoftmax: rank %ld", (long)rank);
  if (axis < 0) axis += rank;
  if (axis < 0 || axis >= rank) DNNRT_FAIL("dnnrtSoftmax: axis out of range");
  if (handle->format != DNNRT_NCHW && rank == 4) DNNRT_FAIL("dnnrtSoftmax: channels-last tensors are not supported");
  int64_t outer = 1, inner = 1;
  const int64_t L = dimX[axis];
  for (int64_t i = 0; i < axis; i++) outer *= dimX[i];
  for (int64_t i = axis + 1; i < rank; i++) inner *= dimX[i];
  if (L < 0 || outer < 0 || inner < 0) DNNRT_FAIL("dnnrtSoftmax: negative dim");
  // an empty batch is no work: nothing is launched and Y is left as it is (the reference's zero-block launches do nothing either)
  if (L == 0 || outer == 0 || inner == 0) return Y;
  if (L > INT32_MAX) DNNRT_FAIL("dnnrtSoftmax: bad dims");
#define SOFTMAX_LAUNCH(T)                                                                           \
  do {                                                                                              \
    if (inner == 1) {                                                                               \
      const int64_t blocks = ceil_div(outer, 4);                                                    \
      if (blocks > INT32_MAX) DNNRT_FAIL("dnnrtSoftmax: too many rows");                            \
      hipLaunchKernelGGL((softmax_rows_kernel<T>), dim3((unsigned)blocks), dim3(256), 0,            \
                         handle->stream, (const T *)X, (T *)Y, outer, (int)L);                      \
    } else {                                                                                        \
      const int64_t blocks = ceil_div(outer * inner, 256);                                          \
      if (blocks > INT32_MAX) DNNRT_FAIL("dnnrtSoftmax: tensor too large");                         \
      hipLaunchKernelGGL((softmax_cols_kernel<T>), dim3((unsigned)blocks), dim3(256), 0,            \
                         handle->stream, (const T *)X, (T *)Y, outer, (int)L, inner);               \
    }                                                                                               \
  } while (0)
  if (dtype == DNNRT_F32) SOFTMAX_LAUNCH(float);
  else if (dtype == DNNRT_F16) SOFTMAX_LAUNCH(__half);
  else DNNRT_FAIL("dnnrtSoftmax: dtype %d", dtype);
#undef SOFTMAX_LAUNCH
  DNNRT_CHECK_LAUNCH("dnnrtSoftmax");
  return Y;
}

void *dnnrtLayerNorm(dnnrtHandle_t handle, const void *X, const int64_t *dimX, int64_t rank,
                     const void *gamma, const void *beta, float eps, void *Y, int32_t dtype) {
  if (!handle) DNNRT_FAIL("dnnrtLayerNorm: null handle");
  if (!X || !Y || !dimX || !gamma || !beta) DNNRT_FAIL("dnnrtLayerNorm: null argument");
  if (rank < 1 || rank > 8) DNNRT_FAIL("dnnrtLayerNorm: rank %ld", (long)rank);
  const int64_t L = dimX[rank - 1], rows = numel(dimX, rank - 1);
  if (L < 0 || rows < 0) DNNRT_FAIL("dnnrtLayerNorm: negative dim");
  // an empty batch is no work: nothing is launched and Y is left as it is (the reference's zero-block launches do nothing either)
  if (L == 0 || rows == 0) return Y;
  if (L > INT32_MAX) DNNRT_FAIL("dnnrtLayerNorm: bad dims");
  const int64_t blocks = ceil_div(rows, 4);
  if (blocks > INT32_MAX) DNNRT_FAIL("dnnrtLayerNorm: too many rows");
  if (dtype == DNNRT_F32 && layernorm_in_registers<float>(handle, X, gamma, beta, Y, rows, L, eps)) {
  } else if (dtype == DNNRT_F16 && layernorm_in_registers<__half>(handle, X, gamma, beta, Y, rows, L, eps)) {
  } else if (dtype == DNNRT_F32)
    hipLaunchKernelGGL((layernorm_kernel<float>), dim3((unsigned)blocks), dim3(256), 0, handle->stream,
                       (const float *)X, (const float *)gamma, (const float *)beta, (float *)Y, rows,
                       (int)L, eps);
  else if (dtype == DNNRT_F16)
    hipLaunchKernelGGL((layernorm_kernel<__half>), dim3((unsigned)blocks), dim3(256), 0, handle->stream,
                       (const __half *)X, (const __half *)gamma, (const __half *)beta, (__half *)Y,
                       rows, (int)L, eps);
  else DNNRT_FAIL("dnnrtLayerNorm: dtype %d", dtype);
  DNNRT_CHECK_LAUNCH("dnnrtLayerNorm");
  return Y;
}

}  // extern "C"
