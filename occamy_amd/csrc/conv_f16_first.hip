// fp16 first layers other than the 7x7 one of the ImageNet ResNets: N,C,H,W
// input with at most four channels, a filter of at most 3x3 (any stride and
// padding), 16 to 64 filters, channels-last output (a MobileNetV2's 3 -> 32,
// 3x3, stride 2; a VGG's 3 -> 64, 3x3).
//
// A wavefront owns 32 neighbouring output pixels of an image at a time; the reduction of at most 36 taps is one to three
// MFMAs for them and 32 filters.  A lane gathers its pixel's taps straight from global memory in the MFMA's order (eight of
// sixteen per step; neighbouring lanes are neighbouring pixels; a tap outside the image is a buffer load past the end, which
// reads zero), those of the next 32 pixels while this one's results are computed.  Filters and bias stay in registers over all of a
// wavefront's pixels.  With one pixel and all its filters per thread (a multiply per tap and filter on the vector units, four
// 16-byte stores 64 bytes apart) 3 -> 32 channels, 224x224 stride 2, batch 64 took 48.5 us, now 31 (2.3 TB/s), 3 -> 64 stride 1 302
// and 140.  What is left: the 2-byte loads, sixteen a lane and 32 pixels, each over four to six cache lines.
#include "conv_f16.h"

namespace dnnrt {

typedef _Float16 fl_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 fl_half4 __attribute__((ext_vector_type(4)));
typedef float fl_floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned fl_uintx4 __attribute__((ext_vector_type(4)));
typedef unsigned fl_uintx2 __attribute__((ext_vector_type(2)));

struct FirstF16Plan {
  int tiles, per_image, per_wave;  // of 32 pixels: all, of an image, for a wavefront
  unsigned magic_per_image, magic_q;
  unsigned inv_c, inv_s;  // t / C = t * inv_c >> 16 for t < 64, and by S
};

// workgroups of four wavefronts that a compute unit's registers hold
constexpr int first_resident(int steps, int k8) { return steps + (k8 + 3) / 4 <= 3 && k8 < 8 ? 4 : steps + (k8 + 3) / 4 <= 4 ? 3 : 2; }

template <int STEPS, int K8>  // 16 * STEPS >= taps, K = 8 * K8 filters
__global__ __launch_bounds__(256, first_resident(STEPS, K8)) void conv_f16_first_kernel(const ConvF16Args a, const FirstF16Plan pl) {
#if __HIP_DEVICE_COMPILE__
  constexpr int K = 8 * K8, MB = (K + 31) / 32, TAPS = 8 * STEPS;  // blocks of matrix rows, a lane's taps
  auto lane_filters = [](int mb) constexpr { return (K - 32 * mb < 32 ? K - 32 * mb : 32) / 2; };  // of a block
  constexpr unsigned OUT = 0x80000000u;  // past the end of every operand
  const int lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // runs of neighbouring workgroups (the grid is a multiple of 8) on one XCD: they share input rows in its L2
  const int wg = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
  const int wg_first = wg * 4 * pl.per_wave, first = wg_first + wave, last = min(wg_first + 4 * pl.per_wave, pl.tiles);
  if (first >= last) return;
  const int PQ = a.P * a.Q, HW = a.H * a.W, taps = a.R * a.S * a.C;

  // The input rows of the workgroup's run of pixels (of its first image) to the caches, a byte of each line: the gathers below
  // have few bytes in flight, and waited for memory four times as long.
  unsigned char touched[2] = {};
  if (pl.per_wave > 1) {
    const int n = div_magic(wg_first, pl.per_image, pl.magic_per_image), t0 = wg_first - n * pl.per_image, t1 = min(t0 + 4 * pl.per_wave, pl.per_image);
    const int h0 = max(div_magic(32 * t0, a.Q, pl.magic_q) * a.sh - a.ph, 0);
    const int h1 = min(div_magic(min(32 * t1, PQ) - 1, a.Q, pl.magic_q) * a.sh - a.ph + a.R, a.H);
    const int bytes = 2 * (h1 - h0) * a.W, lines = (bytes + 63) >> 6;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(a.X) + (int64_t)n * a.C * HW, 0, 2 * a.C * HW, 0x00020000);
#pragma unroll
    for (int i = 0; i < 2; i++) {  // channels as fast as threads go round: c = u % C
      const int u = (int)threadIdx.x + 256 * i, line = (int)((unsigned)u * pl.inv_c >> 16), c = u - line * a.C;
      touched[i] = __builtin_amdgcn_raw_buffer_load_b8(rsrc, line < lines ? 2 * (c * HW + h0 * a.W) + 64 * line : (int)OUT, 0, 0);
    }
  }

  auto tap_rs = [&](int t) { return (int)((unsigned)t * pl.inv_c >> 16); };
  unsigned tap_off[TAPS];  // byte offset of a tap
#pragma unroll
  for (int i = 0; i < TAPS; i++) {
    const int t = 16 * (i >> 3) + 8 * half + (i & 7), rs = tap_rs(t), r = (int)((unsigned)rs * pl.inv_s >> 16);
    tap_off[i] = t < taps ? 2u * (unsigned)((t - rs * a.C) * HW + r * a.W + rs - r * a.S) : OUT;
  }

  unsigned short raw[TAPS] = {};
  int next_n = 0, next_pq = 0;
  // Matrix row 8 q + 4 h + i of block mb is filter 32 mb + h F + 4 q + i, F the block's filters of a lane: a lane gets F in order.
  fl_half8 wa[MB][STEPS];
  float bias[MB][16];
  const _Float16 *__restrict__ Wg = reinterpret_cast<const _Float16 *>(a.Wt);  // K x R x S x C
  const _Float16 *__restrict__ biasg = reinterpret_cast<const _Float16 *>(a.bias);
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const int F = lane_filters(mb), at = 4 * (l32 >> 3) + (l32 & 3), f = 32 * mb + (l32 >> 2 & 1) * F + at;
#pragma unroll
    for (int st = 0; st < STEPS; st++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int t = 16 * st + 8 * half + j;
        const bool ok = t < taps && at < F;
        const _Float16 v = Wg[ok ? f * taps + t : 0];
        wa[mb][st][j] = ok ? v : (_Float16)0.f;
      }
#pragma unroll
    for (int e = 0; e < F; e++) bias[mb][e] = biasg ? (float)biasg[32 * mb + half * F + e] : 0.f;
  }
  asm volatile("" ::"v"((unsigned)touched[0]), "v"((unsigned)touched[1]));
  for (int next = first; next < last + 4; next += 4) {  // `next` is requested and, from the second turn on, the one before computed
    const int n = next_n, pq = next_pq;
    fl_floatx16 acc[MB] = {};
#pragma unroll
    for (int st = 0; st < STEPS; st++) {
      fl_half8 x;
#pragma unroll
      for (int j = 0; j < 8; j++) x[j] = __builtin_bit_cast(_Float16, raw[8 * st + j]);
#pragma unroll
      for (int mb = 0; mb < MB; mb++) acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wa[mb][st], x, acc[mb], 0, 0, 0);
    }
    if (next < last) {
      next_n = div_magic(next, pl.per_image, pl.magic_per_image);
      next_pq = 32 * (next - next_n * pl.per_image) + l32;
      const int p = div_magic(next_pq, a.Q, pl.magic_q), q = next_pq - p * a.Q;
      const int ih = p * a.sh - a.ph, iw = q * a.sw - a.pw;
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(a.X) + (int64_t)next_n * a.C * HW, 0, 2 * a.C * HW, 0x00020000);
      const unsigned at = 2u * (unsigned)(ih * a.W + iw);
      const bool inside = next_pq < PQ && ih >= 0 && ih + a.R <= a.H && iw >= 0 && iw + a.S <= a.W;
      if (__all(inside)) {
#pragma unroll
        for (int i = 0; i < TAPS; i++) raw[i] = __builtin_amdgcn_raw_buffer_load_b16(rsrc, (int)(at + tap_off[i]), 0, 0);
      } else {
        int h8 = 8 * half;
        asm volatile("" : "+v"(h8));  // or the taps' rows and columns would be kept in registers over the loop
#pragma unroll
        for (int i = 0; i < TAPS; i++) {
          const int rs = tap_rs(16 * (i >> 3) + h8 + (i & 7)), r = (int)((unsigned)rs * pl.inv_s >> 16), s = rs - r * a.S;
          const bool ok = next_pq < PQ && (unsigned)(ih + r) < (unsigned)a.H && (unsigned)(iw + s) < (unsigned)a.W;
          raw[i] = __builtin_amdgcn_raw_buffer_load_b16(rsrc, (int)(ok ? at + tap_off[i] : OUT), 0, 0);
        }
      }
    }
    if (next == first) continue;
    const auto y_rsrc = __builtin_amdgcn_make_buffer_rsrc(a.Y + (int64_t)n * PQ * K, 0, 2 * PQ * K, 0x00020000);
    // Z may be Y itself: a wavefront reads its elements, then writes them
    const auto z_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(a.Z) + (int64_t)n * PQ * K, 0, a.Z ? 2 * PQ * K : 0, 0x00020000);
    fl_uintx2 out[MB][4];  // four filters each
    by_act_mode(a.act, [&](auto mode_c) {  // one copy per activation mode, picked once
      constexpr int MODE = decltype(mode_c)::value;
#pragma unroll
      for (int mb = 0; mb < MB; mb++) {
        const int F = lane_filters(mb);
        const unsigned at = pq < PQ ? 2u * (unsigned)(pq * K + 32 * mb + half * F) : OUT;
#pragma unroll
        for (int e0 = 0; e0 < F; e0 += 4) {
          fl_half4 z = {}, o;
          if (a.Z) z = __builtin_bit_cast(fl_half4, __builtin_amdgcn_raw_buffer_load_b64(z_rsrc, (int)(at + 2u * e0), 0, 0));
#pragma unroll
          for (int i = 0; i < 4; i++) {
            float v = acc[mb][e0 + i] + bias[mb][e0 + i];
            if (a.Z) v = (float)(_Float16)v + (float)z[i];
            o[i] = (_Float16)apply_act(v, MODE, a.act_coef);
          }
          out[mb][e0 / 4] = __builtin_bit_cast(fl_uintx2, o);
        }
      }
    });
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      const int F = lane_filters(mb);
      if (F == 16) {
        // 64 bytes of each pixel: lanes 16 .. 31 of a half swap the first 16 bytes with lanes 0 .. 15's second, so that a store
        // writes all 64 of 16 pixels (half of 32 pixels' lines a store otherwise)
        const int px = pq & ~31;
#pragma unroll
        for (int d = 0; d < 4; d++) {
          const auto s = __builtin_amdgcn_permlane16_swap(out[mb][d >> 1][d & 1], out[mb][2 + (d >> 1)][d & 1], false, false);
          out[mb][d >> 1][d & 1] = s[0];
          out[mb][2 + (d >> 1)][d & 1] = s[1];
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
          const int mine = px + 16 * t + (l32 & 15);
          const unsigned at = mine < PQ ? 2u * (unsigned)(mine * K + 32 * mb + 16 * half + 8 * (l32 >> 4)) : OUT;
          const fl_uintx4 v = {out[mb][2 * t][0], out[mb][2 * t][1], out[mb][2 * t + 1][0], out[mb][2 * t + 1][1]};
          __builtin_amdgcn_raw_buffer_store_b128(v, y_rsrc, (int)at, 0, 0);
        }
      } else {
        const unsigned at = pq < PQ ? 2u * (unsigned)(pq * K + 32 * mb + half * F) : OUT;
#pragma unroll
        for (int e0 = 0; e0 < F; e0 += 8) {
          if (F % 8 == 0) {
            const fl_uintx4 v = {out[mb][e0 / 4][0], out[mb][e0 / 4][1], out[mb][e0 / 4 + 1][0], out[mb][e0 / 4 + 1][1]};
            __builtin_amdgcn_raw_buffer_store_b128(v, y_rsrc, (int)(at + 2u * e0), 0, 0);
          } else {
            __builtin_amdgcn_raw_buffer_store_b64(out[mb][e0 / 4], y_rsrc, (int)(at + 2u * e0), 0, 0);
            if (e0 + 4 < F) __builtin_amdgcn_raw_buffer_store_b64(out[mb][e0 / 4 + 1], y_rsrc, (int)(at + 2u * e0 + 8), 0, 0);
          }
        }
      }
    }
  }
#endif
}

// Launches the kernel if the problem is one of its shapes; `launched` says whether it did.
bool launch_conv_f16_first(const dnnrtContext *ctx, const ConvF16Args &a, bool &launched) {
  launched = false;
  auto aligned = [](const void *p, uintptr_t to) { return (reinterpret_cast<uintptr_t>(p) & (to - 1)) == 0; };
  const int64_t PQ = (int64_t)a.P * a.Q, per_image = ceil_div(PQ, 32), tiles = a.N * per_image;
  if (a.format != DNNRT_NCHW_TO_NHWC || a.group != 1 || a.C > 4 || a.R > 3 || a.S > 3 || a.K % 8 != 0 || !aligned(a.Y, 16) ||
      !aligned(a.Z, 16) || tiles >= (1ll << 30) || (int64_t)a.C * a.H * a.W >= (1ll << 29) || PQ * a.K >= (1ll << 29) || tiles == 0)
    return true;
  FirstF16Plan pl{};
  pl.tiles = (int)tiles;
  pl.per_image = (int)per_image;
  pl.magic_per_image = magic_of(pl.per_image);
  pl.magic_q = magic_of(a.Q);
  pl.inv_c = (65536 + (unsigned)a.C - 1) / (unsigned)a.C;
  pl.inv_s = (65536 + (unsigned)a.S - 1) / (unsigned)a.S;
  const int steps = (int)ceil_div(a.R * a.S * a.C, 16);
  // as many wavefronts as stay resident at once, each with its share of the pixels
  pl.per_wave = (int)ceil_div(tiles, (int64_t)ctx->num_cu * 4 * first_resident(steps, a.K / 8));
  const unsigned grid = (unsigned)(ceil_div(ceil_div(tiles, 4 * pl.per_wave), 8) * 8);
#define FIRST_STEPS(S_, K8_) \
  case S_: hipLaunchKernelGGL((conv_f16_first_kernel<S_, K8_>), dim3(grid), dim3(256), 0, ctx->stream, a, pl); break
#define FIRST_CASE(K8_) \
  case K8_: switch (steps) { FIRST_STEPS(1, K8_); FIRST_STEPS(2, K8_); FIRST_STEPS(3, K8_); default: return true; } break
  switch (a.K / 8) {
    FIRST_CASE(2); FIRST_CASE(3); FIRST_CASE(4); FIRST_CASE(6); FIRST_CASE(8);
    default: return true;
  }
#undef FIRST_CASE
#undef FIRST_STEPS
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("conv(fp16 first layer): launch failed: %s", hipGetErrorString(e)); return false; }
  launched = true;
  return true;
}

}  // namespace dnnrt
