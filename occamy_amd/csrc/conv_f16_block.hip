// An inverted residual block in one launch, fp16 channels-last: 1x1 expansion (+ bias, activation), 3x3 depthwise
// convolution (+ bias, activation), 1x1 projection (+ bias, residual, activation).  The two tensors between them, six
// times as wide as the block's input and most of what a MobileNetV2 moves, stay in LDS.
//
// A workgroup of G wavefronts owns up to 64 output pixels of one image (TH x TW).  The part of its input patch (the tile
// and the halo of the depthwise windows) that lies in the image goes to LDS once.  The hidden channels are walked over in
// rounds of 32 per wavefront:
//   expand   each wavefront its own 32 channels over the whole patch (MFMA), with bias and activation rounded to fp16 into
//            a slab of its own, [pixel][channel]; pixels outside the image are zeros, the depthwise padding.  No barrier:
//            only this wavefront reads the slab.
//   depthwise  lane = eight channels of a square of 2 x 2 output pixels: 16 reads of the slab serve four windows of nine, and
//            the lane's 72 filter values are read once a round (a pixel per lane with the filters broadcast made LDS the
//            bottleneck: 115 reads and writes a round instead of 70; as scalar loads the filters were waited for eight times).
//            Results replace the slab.
//   project  after a barrier, the G slabs are the right operand of the projection: blocks of 32 output channels x 32 pixels
//            dealt over the wavefronts, accumulators kept over the rounds.
// Values are rounded where the three separate calls round them, from fp32 sums that start at the bias.  The two 1x1 filters
// are read in blocks of 32 rows and 8 columns (512 contiguous bytes), the order the executor uploads them in: rows of the
// plain matrix would cost a cache line per lane and load, and took longer than everything else.
//
// Where the tiles are few the hidden channels are also cut over workgroups (gridDim.z): partial sums through the handle's
// scratch, the last to arrive adds them in order.
//
// What bounds it: where tiles are many, vector instructions (24 -> 144 -> 24 at 56x56, three wavefronts per SIMD: a round of 7500
// cycles is 650 of them a wavefront, the depthwise sums 288) or, with stride 2, the LDS of a tile's slabs, which leaves one and
// a half wavefronts per SIMD; where they are few, the chain of a launch: 3500 cycles until the patch is there, 2500 for the
// filters, 5000 to 8000 a round, 3000 for the result, 6000 to 11000 for a hand-over (160 -> 960 -> 160 at 7x7, batch 64, four parts).
//
// Measured against the three calls at batch 64 (us): 16 -> 96 -> 24 channels, 112x112 stride 2: 104 -> 53; 24 -> 144 -> 24 at
// 56x56: 85 -> 42; 24 -> 144 -> 32 stride 2: 52 -> 28.5; 32 -> 192 -> 32 at 28x28: 34 -> 17; 64 -> 384 -> 64 at 14x14: 34 -> 15;
// 96 -> 576 -> 96: 38 -> 22; 32 -> 16 behind a depthwise layer at 112x112, no expansion: 49 -> 36; 160 -> 960 -> 160 at 7x7 30 -> 19
// (30.5 uncut).  MobileNetV2 with whole channels only and as it is: batch 1 249 -> 211, 8 315 -> 249, 32 378 -> 343, 64 485 -> 444.
#include "conv_f16.h"
#include "dnnrt_exec.h"
#include "partials.h"

#include <algorithm>
#include <cmath>

namespace dnnrt {

bool block_f32_applies(const dnnrtContext *ctx, const dnnrtExecBlock &k);  // conv_f32_block.hip
bool launch_block_f32(const dnnrtContext *ctx, const dnnrtExecBlock &k);

// The handle's ring of cuts, for both types.
const dnnrtBlockCut *find_block_cut(const dnnrtContext *ctx, const int64_t (&sizes)[11]) {
  constexpr unsigned KEPT = sizeof(ctx->block_cuts) / sizeof(ctx->block_cuts[0]);
  for (unsigned i = 0; i < std::min(ctx->block_cuts_found, KEPT); i++)
    if (std::equal(sizes, sizes + 11, ctx->block_cuts[i].sizes)) return &ctx->block_cuts[i];
  return nullptr;
}
void keep_block_cut(const dnnrtContext *ctx, const int64_t (&sizes)[11], dnnrtBlockCut cut) {
  constexpr unsigned KEPT = sizeof(ctx->block_cuts) / sizeof(ctx->block_cuts[0]);
  std::copy(sizes, sizes + 11, cut.sizes);
  ctx->block_cuts[ctx->block_cuts_found % KEPT] = cut;
  ctx->block_cuts_found = ctx->block_cuts_found + 1 < 2 * KEPT ? ctx->block_cuts_found + 1 : KEPT;  // stays past KEPT once it is there
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

struct BlockF16Args {
  const _Float16 *X, *W1, *b1, *Wd, *bd, *W3, *b3, *Z;  // b1, bd, b3, Z may be null; Z is laid out like Y
  _Float16 *Y;
  int N, H, W, Cin, Ch, P, Q, Cout, ph, pw;
  int TH, TW, QH, QW, PH, PW;      // tile, its 2 x 2 squares, its patch
  int xs_bytes, slab_bytes, xrow;  // LDS: input patch, a wavefront's slab; bytes of an input pixel
  int tiles_w, tiles_hw, tiles, per_xcd, blocks_y;  // blocks_y: blocks of 32 output channels per workgroup
  int per_split, part_px;          // groups of 32 hidden channels of a part (gridDim.z of them); pixels of a partial tile
  unsigned magic_tiles_w, magic_tiles_hw, magic_qw, magic_c8;
  unsigned lo1, hi1, lod, hid;  // the inner activations as clamps, twice in a word
  float lo, hi;
};

// max(lo, min(v, hi)) with NaN kept, as the separate calls' comparisons keep it
__device__ __forceinline__ half2v clamp_pair(half2v v, unsigned lo2, unsigned hi2) {
  return __builtin_elementwise_minimum(__builtin_elementwise_maximum(v, __builtin_bit_cast(half2v, lo2)), __builtin_bit_cast(half2v, hi2));
}
// sum += (half xh of x) * (half wh of w).  Written out: from fmaf() of converted values that several sums share, the compiler
// keeps all 72 filter values converted, in registers that then spill.
__device__ __forceinline__ void fma_halves(float &sum, unsigned x, int xh, unsigned w, int wh) {
  if (xh == 0 && wh == 0) asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel_hi:[1,1,0]" : "+v"(sum) : "v"(x), "v"(w));
  else if (xh == 1 && wh == 0) asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[1,0,0] op_sel_hi:[1,1,0]" : "+v"(sum) : "v"(x), "v"(w));
  else if (xh == 0) asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[0,1,0] op_sel_hi:[1,1,0]" : "+v"(sum) : "v"(x), "v"(w));
  else asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "+v"(sum) : "v"(x), "v"(w));
}
__device__ __forceinline__ unsigned dword(half8 v, int i) {
  typedef unsigned uint4v __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(uint4v, v)[i];
}
constexpr int SLAB_PX = 80;  // bytes of a slab's pixel: 32 channels, and 16 against bank conflicts (96 has fewer, but 56x56 stride 2: 54 us -> 65)
// A barrier that waits for this wavefront's LDS accesses but not for its loads from global memory.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// S: the depthwise stride.  KC: steps of 16 input channels (0: no expansion, X holds the hidden channels).  GM: most
// wavefronts of a workgroup.  PARTS: the hidden channels are cut over workgroups; kernels of whole channels go without the hand-over, whose
// operands cost them scalar registers (MobileNetV2 at batch 64: 470 us with it in every kernel, 464 without).
template <int S, int KC, int GM, bool PARTS>
__global__ __launch_bounds__(64 * GM) __attribute__((amdgpu_waves_per_eu(KC <= 2 ? 3 : 2))) void conv_f16_block_kernel(const BlockF16Args a, float *partials,
                                                                                                                       unsigned *counters) {
  constexpr bool EXPAND = KC > 0;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = (int)(blockDim.x >> 6);
  char *Xs = smem, *slabs = smem + a.xs_bytes, *mine = slabs + wave * a.slab_bytes;
  // this workgroup's groups of 32 hidden channels: from group0 on
  const int group0 = PARTS ? (int)blockIdx.z * a.per_split : 0, groups = min(a.per_split, ((a.Ch + 31) >> 5) - group0);
  float *B1 = reinterpret_cast<float *>(slabs + G * a.slab_bytes), *Bd = B1 + 32 * groups;  // the inner biases, padded to the last group's end
  _Float16 *Wd = reinterpret_cast<_Float16 *>(Bd + 32 * groups);  // the depthwise filters, [channel][tap]

  const int b = (int)blockIdx.x, tile = (b & 7) * a.per_xcd + (b >> 3);  // neighbouring tiles share their halo in one XCD's L2
  if (tile >= a.tiles) return;
  const int n = div_magic(tile, a.tiles_hw, a.magic_tiles_hw), tr = tile - n * a.tiles_hw;
  const int ty = div_magic(tr, a.tiles_w, a.magic_tiles_w);
  const int p0 = ty * a.TH, q0 = (tr - ty * a.tiles_w) * a.TW;
  const int h0 = p0 * S - a.ph, w0 = q0 * S - a.pw;
  // the patch's part in the image: RH x RW pixels from (r0, c0) of the patch on
  const int r0 = max(0, -h0), c0 = max(0, -w0);
  const int RH = min(a.PH, a.H - h0) - r0, RW = min(a.PW, a.W - w0) - c0, NP = RH * RW;
  const unsigned inv_rw = (65536u + RW - 1) / (unsigned)RW;  // px / RW = px * inv_rw >> 16 for px < 1024
  const bool border = RH < a.PH || RW < a.PW;
  const _Float16 *Xn = a.X + ((int64_t)n * a.H * a.W + (h0 + r0) * a.W + w0 + c0) * a.Cin;
  auto row_of = [&](int px) { return (int)((unsigned)px * inv_rw >> 16); };
  const half8 zero8 = {};

  // Buffer loads here and below: what lies past an operand reads as zeros without a mask or a branch behind the load, either
  // of which is a wait for it.
  constexpr unsigned OUT = 0x80000000u;
  auto rsrc_of = [](const _Float16 *w, int n) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(w), 0, w ? 2 * n : 0, 0x00020000); };
  // The input patch, the depthwise filters and the inner biases to LDS: everything is requested before anything is stored
  // (as loops of load and store, four to six times the latency of memory before the first product).
  {
    const int from = 32 * group0;
    const auto x_rsrc = rsrc_of(Xn, a.H * a.W * a.Cin), wd_rsrc = rsrc_of(a.Wd + 9 * from, 9 * (a.Ch - from));
    const auto b1_rsrc = rsrc_of(a.b1 ? a.b1 + from : nullptr, a.Ch - from), bd_rsrc = rsrc_of(a.bd ? a.bd + from : nullptr, a.Ch - from);
    constexpr int XU = EXPAND ? 6 : 0, WU = 3, BU = 3;
    const int c8n = a.Cin >> 3, x_units = EXPAND ? NP * c8n : 0, w_units = 36 * groups, b_units = 32 * groups, step = 64 * G;
    for (int x0 = tid, w0 = tid, b0 = tid; x0 < x_units || w0 < w_units || b0 < b_units; x0 += XU * step, w0 += WU * step, b0 += BU * step) {
      half8 xv[XU > 0 ? XU : 1], wv[WU];
      unsigned short b1v[BU], bdv[BU];
#pragma unroll
      for (int i = 0; i < XU; i++) {
        const int u = x0 + i * step, px = div_magic(u, c8n, a.magic_c8), c = u - px * c8n, r = row_of(px);
        xv[i] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, u < x_units ? (unsigned)(2 * ((r * a.W + px - r * RW) * a.Cin + 8 * c)) : OUT, 0, 0));
      }
#pragma unroll
      for (int i = 0; i < WU; i++) wv[i] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(wd_rsrc, 16 * (w0 + i * step), 0, 0));
#pragma unroll
      for (int i = 0; i < BU; i++) {
        b1v[i] = __builtin_amdgcn_raw_buffer_load_b16(b1_rsrc, 2 * (b0 + i * step), 0, 0);
        bdv[i] = __builtin_amdgcn_raw_buffer_load_b16(bd_rsrc, 2 * (b0 + i * step), 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < XU; i++) {
        const int u = x0 + i * step, px = div_magic(u, c8n, a.magic_c8), c = u - px * c8n;
        if (u < x_units) *reinterpret_cast<half8 *>(Xs + px * a.xrow + 16 * c) = xv[i];
      }
#pragma unroll
      for (int i = 0; i < WU; i++)
        if (w0 + i * step < w_units) *reinterpret_cast<half8 *>(Wd + 8 * (w0 + i * step)) = wv[i];
#pragma unroll
      for (int i = 0; i < BU; i++) {
        if (b0 + i * step >= b_units) continue;
        B1[b0 + i * step] = (float)__builtin_bit_cast(_Float16, b1v[i]);
        Bd[b0 + i * step] = (float)__builtin_bit_cast(_Float16, bdv[i]);
      }
    }
  }
  // depthwise: lane = eight channels of a 2 x 2 square of output pixels (squares past the tile repeat its first)
  const int cg = lane & 3, square = (lane >> 2) < a.QH * a.QW ? lane >> 2 : 0;
  const int sy = div_magic(square, a.QW, a.magic_qw), sx = square - sy * a.QW;
  const char *win = mine + (2 * sy * S * a.PW + 2 * sx * S) * SLAB_PX + 16 * cg;

  // A 1x1 filter's rows 32 g .. + 31 at columns col .. col + 7, from the blocked layout.
  auto load_rows = [&](__amdgpu_buffer_rsrc_t w, int rows, int cols, int g, int col) -> half8 {
    const int in = min(32, rows - 32 * g);
    const unsigned at = col < cols && l32 < in ? (unsigned)(2 * (32 * g * cols + ((col >> 3) * in + l32) * 8)) : OUT;
    return __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(w, at, 0, 0));
  };
  const auto w1_rsrc = rsrc_of(a.W1, a.Ch * a.Cin), w3_rsrc = rsrc_of(a.W3, a.Cout * a.Ch);
  [[maybe_unused]] half8 wa[EXPAND ? KC : 1];
  auto load_expand = [&](int g) {
    if constexpr (EXPAND)
#pragma unroll
      for (int k = 0; k < KC; k++) wa[k] = load_rows(w1_rsrc, a.Ch, a.Cin, g, 16 * k + 8 * half);
  };
  load_expand(group0 + min(wave, groups - 1));

  // projection: a wavefront's block of 32 output channels; its 32 pixels of the tile, or all 64 where the wavefronts do not
  // suffice for twice the blocks
  const int mfirst = (int)blockIdx.y * a.blocks_y, mblocks = min(a.blocks_y, ((a.Cout + 31) >> 5) - mfirst);
  const bool pairs = 2 * mblocks <= G;
  const int pm = pairs ? wave >> 1 : wave, ppx = pairs ? 32 * (wave & 1) : 0;
  floatx16 acc[2];
  {
    const auto b3_rsrc = rsrc_of(!PARTS || blockIdx.z == 0 ? a.b3 : nullptr, a.Cout);  // in the first part's sums
#pragma unroll
    for (int gq = 0; gq < 4; gq++) {
      const half4 v = __builtin_bit_cast(half4, __builtin_amdgcn_raw_buffer_load_b64(b3_rsrc, 2 * (32 * (mfirst + pm) + 8 * gq + 4 * half), 0, 0));
#pragma unroll
      for (int i = 0; i < 4; i++) acc[0][4 * gq + i] = acc[1][4 * gq + i] = (float)v[i];
    }
  }
  __syncthreads();

  for (int first = 0; first < groups; first += G) {
    const int g = first + wave, ch = 32 * (group0 + g), own = 32 * g;  // hidden channels; theirs among the workgroup's
    // The projection's filter for this round: half of it is requested well ahead where there are registers for that (all of it took more than
    // there are, and scratch memory; 7x7 blocks of 160 channels, which have none to spare: with half ahead as fast).
    constexpr int EARLY = KC <= 2 || KC > 8 ? 0 : GM / 2;
    half8 wp[2 * GM];
    auto load_project = [&](int from, int to) {
#pragma unroll
      for (int q = 0; q < GM; q++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const int c = 32 * (group0 + first + q) + 16 * k + 8 * half;
          if (q >= from && q < to) wp[2 * q + k] = load_rows(w3_rsrc, a.Cout, a.Ch, mfirst + min(pm, mblocks - 1), q < G ? c : a.Ch);
        }
    };
    load_project(0, EARLY);
    if (g < groups) {
      if (border)
        for (int u = lane; u < a.PH * a.PW * (SLAB_PX / 16); u += 64) *reinterpret_cast<half8 *>(mine + 16 * u) = zero8;
      // ---- expand ---------------------------------------------------------------
      if constexpr (EXPAND) {
        floatx16 bias;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float4 v = *reinterpret_cast<const float4 *>(B1 + own + 8 * q + 4 * half);
          bias[4 * q] = v.x; bias[4 * q + 1] = v.y; bias[4 * q + 2] = v.z; bias[4 * q + 3] = v.w;
        }
        for (int p = 0; p < NP; p += 32) {
          const int px = p + l32, pc = min(px, NP - 1), r = row_of(pc);
          const char *xp = Xs + pc * a.xrow;
          floatx16 e = bias;
#pragma unroll
          for (int k = 0; k < KC; k++) {
            const int c = 16 * k + 8 * half;
            half8 v = *reinterpret_cast<const half8 *>(xp + 2 * min(c, a.Cin - 8));
            v = c < a.Cin ? v : zero8;
            e = __builtin_amdgcn_mfma_f32_32x32x16_f16(wa[k], v, e, 0, 0, 0);
          }
          const int at = (r0 + r) * a.PW + c0 + pc - r * RW;
#pragma unroll
          for (int q = 0; q < 4; q++) {
            uint2 o;
            o.x = __builtin_bit_cast(unsigned, clamp_pair(half2v{(_Float16)e[4 * q], (_Float16)e[4 * q + 1]}, a.lo1, a.hi1));
            o.y = __builtin_bit_cast(unsigned, clamp_pair(half2v{(_Float16)e[4 * q + 2], (_Float16)e[4 * q + 3]}, a.lo1, a.hi1));
            if (px < NP) *reinterpret_cast<uint2 *>(mine + at * SLAB_PX + 16 * q + 8 * half) = o;
          }
        }
        load_expand(group0 + min(g + G, groups - 1));
      } else {
        for (int u = lane; u < NP * 4; u += 64) {
          const int px = u >> 2, q = u & 3, r = row_of(px), c = ch + 8 * q;
          const half8 v = *reinterpret_cast<const half8 *>(Xn + (r * a.W + px - r * RW) * a.Cin + min(c, a.Ch - 8));
          *reinterpret_cast<half8 *>(mine + ((r0 + r) * a.PW + c0 + px - r * RW) * SLAB_PX + 16 * q) = v;
        }
      }
      asm volatile("" ::: "memory");  // a wavefront's LDS accesses stay in order
      // ---- depthwise --------------------------------------------------------------
      constexpr int WIN = 3 + S;  // rows and columns of input under a square
      half8 w[9];  // filter e of the eight, tap t: value 9 e + t
#pragma unroll
      for (int i = 0; i < 9; i++) w[i] = *reinterpret_cast<const half8 *>(Wd + (own + 8 * cg) * 9 + 8 * i);
      float sum[4][8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float bv = Bd[own + 8 * cg + e];
#pragma unroll
        for (int o = 0; o < 4; o++) sum[o][e] = bv;
      }
#pragma unroll
      for (int r = 0; r < WIN; r++) {
        __builtin_amdgcn_sched_barrier(0);  // a row's values at a time: more would not fit the registers
        half8 h[WIN];
#pragma unroll
        for (int c = 0; c < WIN; c++) h[c] = *reinterpret_cast<const half8 *>(win + (r * a.PW + c) * SLAB_PX);
#pragma unroll
        for (int o = 0; o < 4; o++) {
          const int tr = r - (o >> 1) * S;
          if (tr < 0 || tr > 2) continue;
#pragma unroll
          for (int s = 0; s < 3; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
              const int at = 9 * e + 3 * tr + s;
              fma_halves(sum[o][e], dword(h[(o & 1) * S + s], e >> 1), e & 1, dword(w[at >> 3], (at & 7) >> 1), at & 1);
            }
        }
      }
      // all lanes have read their windows: the slab is free for the results, squares' pixels in a row
#pragma unroll
      for (int o = 0; o < 4; o++) {
        uint4 d;
        d.x = __builtin_bit_cast(unsigned, clamp_pair(half2v{(_Float16)sum[o][0], (_Float16)sum[o][1]}, a.lod, a.hid));
        d.y = __builtin_bit_cast(unsigned, clamp_pair(half2v{(_Float16)sum[o][2], (_Float16)sum[o][3]}, a.lod, a.hid));
        d.z = __builtin_bit_cast(unsigned, clamp_pair(half2v{(_Float16)sum[o][4], (_Float16)sum[o][5]}, a.lod, a.hid));
        d.w = __builtin_bit_cast(unsigned, clamp_pair(half2v{(_Float16)sum[o][6], (_Float16)sum[o][7]}, a.lod, a.hid));
        *reinterpret_cast<uint4 *>(mine + (4 * (lane >> 2) + o) * SLAB_PX + 16 * cg) = ch + 8 * cg < a.Ch ? d : make_uint4(0, 0, 0, 0);
      }
    }
    load_project(EARLY, GM);
    lds_barrier();

    // ---- project ------------------------------------------------------------------
    if (pm < mblocks) {
#pragma unroll
      for (int q = 0; q < GM; q++) {
        if (q < G && first + q < groups) {
#pragma unroll
          for (int k = 0; k < 2; k++) {
            const char *at = slabs + q * a.slab_bytes + (ppx + l32) * SLAB_PX + 32 * k + 16 * half;
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wp[2 * q + k], *reinterpret_cast<const half8 *>(at), acc[0], 0, 0, 0);
            if (!pairs) acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wp[2 * q + k], *reinterpret_cast<const half8 *>(at + 32 * SLAB_PX), acc[1], 0, 0, 0);
          }
        }
      }
    }
    if (first + G < groups) lds_barrier();
  }

  auto place = [&](int px, int &p, int &q) -> bool {  // the tile's pixel px in the image
    const int sq = px >> 2, py = div_magic(sq, a.QW, a.magic_qw);
    p = p0 + 2 * py + (px >> 1 & 1);
    q = q0 + 2 * (sq - py * a.QW) + (px & 1);
    return py < a.QH && p < a.P && q < a.Q;
  };
  // ---- hidden channels cut over workgroups: partial sums through the handle's scratch (igemm_f32_small.hip states what the
  // hand-over rests on), [block of channels][four of them][pixel]; the last to arrive adds the parts in order and goes on
#if __HIP_DEVICE_COMPILE__
  if constexpr (PARTS) {
    const int parts = (int)gridDim.z;
    const __amdgpu_buffer_rsrc_t rsrc = part_rsrc(partials);
    const unsigned slot = blockIdx.y * (unsigned)a.tiles + (unsigned)tile, part_bytes = (unsigned)a.blocks_y * 128u * (unsigned)a.part_px;
    const int across = min(a.TW, a.Q);
    unsigned at[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      int p, q;
      const bool ok = place(ppx + 32 * t + l32, p, q) && pm < mblocks && (t == 0 || !pairs);
      at[t] = ok ? 16u * (unsigned)((pm * 8 + half) * a.part_px + (p - p0) * across + q - q0) : PART_NONE;
    }
    const unsigned step = 32u * (unsigned)a.part_px;  // from four channels of a lane to the next
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int gq = 0; gq < 4; gq++)
        if (t == 0 || !pairs)
          part_store(rsrc, at[t], (slot * parts + blockIdx.z) * part_bytes + gq * step, part_floatx4{acc[t][4 * gq], acc[t][4 * gq + 1], acc[t][4 * gq + 2], acc[t][4 * gq + 3]});
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    volatile unsigned *arrived = reinterpret_cast<unsigned *>(smem);
    if (tid == 0) *arrived = __hip_atomic_fetch_add(&counters[slot], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived != (unsigned)parts - 1) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (tid == 0) __hip_atomic_store(&counters[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[t][r] = 0.f;
    for (int y = 0; y < parts; y += 2) {  // two parts in flight
      part_floatx4 v[2][2][4];
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
          for (int gq = 0; gq < 4; gq++)
            v[u][t][gq] = part_load<part_floatx4>(rsrc, y + u < parts ? at[t] : PART_NONE, (slot * parts + (unsigned)min(y + u, parts - 1)) * part_bytes + gq * step);
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[t][r] += v[u][t][r >> 2][r & 3];
    }
  }
#endif

  // ---- residual, activation: the lane's pixel, four consecutive channels per access ------------------------------
  if (pm >= mblocks) return;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    if (t == 1 && pairs) break;
    int p, q;
    if (!place(ppx + 32 * t + l32, p, q)) continue;
    const int c0y = 32 * (mfirst + pm) + 4 * half;
    const int64_t at = (((int64_t)n * a.P + p) * a.Q + q) * a.Cout + c0y;
    half4 z[4] = {};
    if (a.Z)
#pragma unroll
      for (int gq = 0; gq < 4; gq++) z[gq] = *reinterpret_cast<const half4 *>(a.Z + at + (c0y + 8 * gq < a.Cout ? 8 * gq : 0));
#pragma unroll
    for (int gq = 0; gq < 4; gq++) {
      if (c0y + 8 * gq >= a.Cout) continue;
      half4 out;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float v = acc[t][4 * gq + i];
        if (a.Z) v = (float)(_Float16)v + (float)z[gq][i];
        v = v < a.lo ? a.lo : v;
        out[i] = (_Float16)(v > a.hi ? a.hi : v);
      }
      *reinterpret_cast<half4 *>(a.Y + at + 8 * gq) = out;
    }
  }
}

// ---- which problems, which tile ----------------------------------------------------
static bool clamp_of(int64_t mode, float coef, unsigned &lo2, unsigned &hi2) {
  _Float16 lo, hi;
  lo = mode == DNNRT_ACT_IDENTITY ? (_Float16)-__builtin_inff() : (_Float16)0.f;
  hi = mode == DNNRT_ACT_CLIPPED_RELU ? (_Float16)coef : (_Float16)__builtin_inff();
  lo2 = 0x10001u * __builtin_bit_cast(unsigned short, lo);
  hi2 = 0x10001u * __builtin_bit_cast(unsigned short, hi);
  if (mode == DNNRT_ACT_CLIPPED_RELU) return (float)hi == coef && coef >= 0.f;
  return mode == DNNRT_ACT_IDENTITY || mode == DNNRT_ACT_RELU;
}

constexpr int BLOCK_LDS = 160 * 1024;
constexpr int BLOCK_PER_GROUP = 2 * 32 * 4 + 32 * 9 * 2;  // biases and depthwise filters of 32 hidden channels

// grid_y, G: workgroups per tile, wavefronts per workgroup
// `faster`: refuse what the separate calls do sooner.
static bool plan_block_f16(const dnnrtContext *ctx, const dnnrtExecBlock &k, bool faster, BlockF16Args &a, int &kc, int &grid_y, int &G, int &parts) {
  const int num_cu = ctx->num_cu;
  if (k.dtype != DNNRT_F16 || k.format != DNNRT_NHWC || k.r != 3 || k.s != 3 || (k.stride != 1 && k.stride != 2) || k.cin % 8 || k.ch % 8 || k.cout % 8) return false;
  if (!k.expand && k.cin != k.ch) return false;
  // Every tile's patch must hold a row and a column of the image (the kernel divides by their number, and with none it would
  // compute padding from what lies beside the image): tiles are two pixels or more, so a padding of up to two leaves one.
  if (k.n < 1 || k.h < 1 || k.w < 1 || k.pad_h < 0 || k.pad_h > 2 || k.pad_w < 0 || k.pad_w > 2) return false;
  if (k.h + 2 * k.pad_h < 3 || k.w + 2 * k.pad_w < 3 || k.p != (k.h + 2 * k.pad_h - 3) / k.stride + 1 || k.q != (k.w + 2 * k.pad_w - 3) / k.stride + 1) return false;
  const int64_t lim = 1ll << 29;  // elements of a buffer
  if (k.h * k.w * k.cin > lim || k.p * k.q * k.cout > lim || k.ch * std::max(k.cin, k.cout) > lim || k.n * k.p * k.q > lim || k.ch > 4096 || k.cout > 4096) return false;
  if ((k.expand && !clamp_of(k.act1, k.coef1, a.lo1, a.hi1)) || !clamp_of(k.actd, k.coefd, a.lod, a.hid)) return false;
  if (k.act != DNNRT_ACT_IDENTITY && k.act != DNNRT_ACT_RELU && k.act != DNNRT_ACT_CLIPPED_RELU) return false;
  a.lo = k.act == DNNRT_ACT_IDENTITY ? -__builtin_inff() : 0.f;
  a.hi = k.act == DNNRT_ACT_CLIPPED_RELU ? k.coef : __builtin_inff();
  const int steps = (int)ceil_div(k.cin, 16);
  kc = !k.expand ? 0 : steps <= 1 ? 1 : steps <= 2 ? 2 : steps <= 4 ? 4 : steps <= 6 ? 6 : steps <= 10 ? 10 : -1;
  if (kc < 0) return false;
  a.N = (int)k.n; a.H = (int)k.h; a.W = (int)k.w; a.Cin = (int)k.cin; a.Ch = (int)k.ch; a.P = (int)k.p; a.Q = (int)k.q; a.Cout = (int)k.cout;
  a.ph = (int)k.pad_h; a.pw = (int)k.pad_w;
  a.xrow = k.expand ? 16 * (a.Cin / 8 | 1) : 0;  // an odd number of 16-byte chunks: neighbouring pixels meet no bank twice
  const int mall = (int)ceil_div(a.Cout, 32), groups = (int)ceil_div(a.Ch, 32);
  grid_y = (int)ceil_div(mall, 5);
  a.blocks_y = (int)ceil_div(mall, grid_y);
  const int most = kc <= 2 ? 4 : 8;  // wavefronts, the kernel's GM
  if (a.blocks_y > most) return false;
  // Tile, wavefronts and parts by estimated time, fitted to 6300 cuts of MobileNetV2's twelve kinds of blocks at batch 1, 4, 16, 32
  // and 64, 6 .. 60 us, within 8 % on the whole; the cut it picks takes 3 % more than the best of them on average.  What counts
  // is what a round waits for, less what it computes.
  auto cut = [&](int qw, int g, int n_parts, BlockF16Args &o) -> double {  // microseconds; 0: cannot be
    const int qh = std::min(16 / qw, (a.P + 1) / 2), tw = 2 * qw, th = 2 * qh;
    const int pw = (tw - 1) * (int)k.stride + 3, ph = (th - 1) * (int)k.stride + 3, np = pw * ph;
    const int xs = (int)ceil_div(np, 32) * 32 * a.xrow, slab = std::max(np, 64) * SLAB_PX;
    const int per = (int)ceil_div(groups, n_parts);
    if (ceil_div(groups, per) != n_parts) return 0;
    const int lds = xs + g * slab + BLOCK_PER_GROUP * per;
    if (lds > BLOCK_LDS) return 0;
    const double tiles = (double)a.N * (double)ceil_div(a.P, th) * (double)ceil_div(a.Q, tw) * grid_y, units = tiles * n_parts;
    const int in = std::min(ph, a.H) * std::min(pw, a.W), part_px = std::min(th, a.P) * std::min(tw, a.Q);
    const double part_bytes = a.blocks_y * 128.0 * part_px;
    if (n_parts > 1 && (ctx->splitk_shared || tiles > ctx->splitk_max_tiles || units * part_bytes > (double)ctx->splitk_partial_bytes)) return 0;
    const double rounds = (double)ceil_div(per, g);
    const double per_round = (k.stride == 1 ? 520.0 : 1880.0) + 28.0 * kc * (double)ceil_div(in, 32);  // cycles of a wavefront beside others
    const int per_cu = std::min(160 * 1024 / lds, (kc <= 2 ? 12 : 8) / g);  // two or three wavefronts per SIMD
    if (per_cu < 1) return 0;
    // what a compute unit has at a time, and how long that takes
    const double at_once = std::min((double)per_cu, std::max(1.0, units / num_cu));
    const double turns = std::max(1.0, units / (at_once * num_cu)), turn = rounds * (per_round * at_once * g / 4 + 7560 + 72.0 * kc * g) + 6290;
    o.TH = th; o.TW = tw; o.QH = qh; o.QW = qw; o.PH = ph; o.PW = pw; o.xs_bytes = xs; o.slab_bytes = slab; o.per_split = per; o.part_px = part_px;
    return 0.95 + 0.43 * a.blocks_y + turn * (turns + 0.81 * (std::ceil(turns) - turns)) / 2300 + (n_parts > 1 ? 2.7 + n_parts * part_bytes / 4.4e4 : 0.0);
  };
  const int64_t sizes[11] = {k.n, k.cin, k.h, k.w, k.ch, k.cout, k.stride, k.pad_h, k.pad_w, k.expand + 2 * k.dtype, ctx->splitk_partial_bytes};
  double best = 0;
  if (const dnnrtBlockCut *f = find_block_cut(ctx, sizes)) {
    best = cut(f->qw, f->waves, f->splits, a);
    G = f->waves;
    parts = f->splits;
  }
  if (best == 0) {
    BlockF16Args t = a;
    int best_qw = 0;
    for (int qw = 1; qw <= 16 && (qw == 1 || 2 * (qw - 1) < a.Q); qw++)
      for (int g = std::max(a.blocks_y, k.expand ? 2 : 1); g <= most && (g == a.blocks_y || g <= std::max(groups, 2)); g++)
        for (int n = 1; n <= groups && n <= 32; n++) {
          const double us = cut(qw, g, n, t);
          if (us > 0 && (best == 0 || us < best)) { best = us; best_qw = qw; G = g; parts = n; }
          if ((double)a.N * (double)(ceil_div(a.P, 2 * std::min(16 / qw, (a.P + 1) / 2)) * ceil_div(a.Q, 2 * qw)) * grid_y * n >= 2.0 * num_cu) break;  // enough of them
        }
    if (best == 0) return false;
    cut(best_qw, G, parts, a);
    keep_block_cut(ctx, sizes, dnnrtBlockCut{{}, 0, best_qw, G, parts});
  }
  // What the separate calls take inside a network, in microseconds (MobileNetV2's at batch 1, 8, 16 and 32, within a fifth): a
  // launch each, their megabytes, and the projection's long reduction on few tiles (up to 64 pixels have a kernel of their own).
  const double in_px = (double)a.N * a.H * a.W, out_px = (double)a.N * a.P * a.Q;
  const double mb1 = in_px * (a.Cin + a.Ch) * 2e-6, mbd = (in_px + out_px) * a.Ch * 2e-6, mb3 = out_px * (a.Ch + a.Cout) * 2e-6;
  const double us1 = k.expand ? 3.8 + std::min(1.2, 2 * mb1) + 0.55 * mb1 : 0, usd = 4.8 + 0.35 * mbd;
  const double us3 = 3.6 + (out_px <= 64 ? 0.0015 : 0.0055) * a.Ch + 0.2 * mb3;
  if (faster && best > 0.95 * (us1 + usd + us3)) return false;
  a.tiles_w = (int)ceil_div(a.Q, a.TW);
  a.tiles_hw = a.tiles_w * (int)ceil_div(a.P, a.TH);
  a.tiles = a.N * a.tiles_hw;
  a.per_xcd = (int)ceil_div(a.tiles, 8);
  a.magic_tiles_w = magic_of(a.tiles_w); a.magic_tiles_hw = magic_of(a.tiles_hw); a.magic_qw = magic_of(a.QW); a.magic_c8 = magic_of(std::max(a.Cin / 8, 1));
  return true;
}

bool block_f16_applies(const dnnrtContext *ctx, const dnnrtExecBlock &k) {
  BlockF16Args a{};
  int kc, gy, g, parts;
  return plan_block_f16(ctx, k, true, a, kc, gy, g, parts);
}

template <int S, int KC, int GM, bool PARTS>
static bool launch_one(const dnnrtContext *ctx, dim3 grid, dim3 threads, size_t lds, const BlockF16Args &a) {
  static LdsRaised raised;
  if (!raise_lds(raised, ctx->device, reinterpret_cast<const void *>(&conv_f16_block_kernel<S, KC, GM, PARTS>), BLOCK_LDS)) {
    set_error("inverted residual block (fp16): cannot reserve %d bytes of LDS", BLOCK_LDS);
    return false;
  }
  hipLaunchKernelGGL((conv_f16_block_kernel<S, KC, GM, PARTS>), grid, threads, lds, ctx->stream, a, ctx->splitk_partials, ctx->splitk_counters);
  return true;
}

static bool launch_cut(const dnnrtContext *ctx, const dnnrtExecBlock &k, BlockF16Args &a, int kc, int gy, int g, int parts) {
  a.X = static_cast<const _Float16 *>(k.x); a.W1 = static_cast<const _Float16 *>(k.w1); a.b1 = static_cast<const _Float16 *>(k.b1);
  a.Wd = static_cast<const _Float16 *>(k.wd); a.bd = static_cast<const _Float16 *>(k.bd);
  a.W3 = static_cast<const _Float16 *>(k.w3); a.b3 = static_cast<const _Float16 *>(k.b3);
  a.Z = static_cast<const _Float16 *>(k.z); a.Y = static_cast<_Float16 *>(k.y);
  for (const void *q : {k.x, k.w1, k.b1, k.wd, k.bd, k.w3, k.b3, k.z, (const void *)k.y})
    if (!aligned16(q)) { set_error("inverted residual block (fp16): an operand is not 16-byte aligned"); return false; }
  const dim3 grid((unsigned)(8 * a.per_xcd), (unsigned)gy, (unsigned)parts), threads(64 * (unsigned)g);
  const size_t lds = (size_t)a.xs_bytes + (size_t)g * (size_t)a.slab_bytes + BLOCK_PER_GROUP * (size_t)a.per_split;
#define BLOCK(S, KC)                                                                        \
  if (!(parts > 1 ? launch_one<S, KC, KC <= 2 ? 4 : 8, true>(ctx, grid, threads, lds, a)    \
                  : launch_one<S, KC, KC <= 2 ? 4 : 8, false>(ctx, grid, threads, lds, a))) \
  return false
  if (k.stride == 1) switch (kc) {
    case 0: BLOCK(1, 0); break; case 1: BLOCK(1, 1); break; case 2: BLOCK(1, 2); break;
    case 4: BLOCK(1, 4); break; case 6: BLOCK(1, 6); break; default: BLOCK(1, 10); break;
  } else switch (kc) {
    case 0: BLOCK(2, 0); break; case 1: BLOCK(2, 1); break; case 2: BLOCK(2, 2); break;
    case 4: BLOCK(2, 4); break; case 6: BLOCK(2, 6); break; default: BLOCK(2, 10); break;
  }
#undef BLOCK
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("inverted residual block (fp16): launch failed: %s", hipGetErrorString(e)); return false; }
  return true;
}

bool launch_block_f16(const dnnrtContext *ctx, const dnnrtExecBlock &k) {
  BlockF16Args a{};
  int kc, gy, g, parts;
  if (!plan_block_f16(ctx, k, false, a, kc, gy, g, parts)) { set_error("inverted residual block (fp16): not a shape this kernel takes"); return false; }
  return launch_cut(ctx, k, a, kc, gy, g, parts);
}

}  // namespace dnnrt

extern "C" {

int32_t dnnrtExecBlockApplies(dnnrtHandle_t handle, const dnnrtExecBlock *block) {
  return handle && block && (block->dtype == DNNRT_F32 ? dnnrt::block_f32_applies(handle, *block) : dnnrt::block_f16_applies(handle, *block)) ? 1 : 0;
}

void dnnrtExecBlockFilter(void *dst, const void *src, int64_t rows, int64_t cols) {
  const uint16_t *from = static_cast<const uint16_t *>(src);
  uint16_t *to = static_cast<uint16_t *>(dst);
  for (int64_t r0 = 0; r0 < rows; r0 += 32)
    for (int64_t c = 0; c < cols; c += 8)
      for (int64_t r = r0; r < rows && r < r0 + 32; r++)
        for (int64_t i = 0; i < 8; i++) *to++ = from[r * cols + c + i];
}

int32_t dnnrtExecRunBlock(dnnrtHandle_t handle, const dnnrtExecBlock *block) {
  if (!handle || !block || !block->x || !block->wd || !block->w3 || !block->y || (block->expand && !block->w1)) {
    dnnrt::set_error("dnnrtExecRunBlock: bad arguments");
    return 1;
  }
  return (block->dtype == DNNRT_F32 ? dnnrt::launch_block_f32(handle, *block) : dnnrt::launch_block_f16(handle, *block)) ? 0 : 1;
}

}  // extern "C"
