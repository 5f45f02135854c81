// An inverted residual block in one launch, fp32 N,C,H,W: 1x1 expansion (+ bias, activation), 3x3
// depthwise convolution (+ bias, activation), 1x1 projection (+ bias, residual, activation).  The two tensors between them,
// six times as wide as the block's input, stay in LDS.
//
// A workgroup of G wavefronts owns a tile of up to 16 NB output pixels of one image, 2 x 2 squares of them, and a range of the
// hidden channels.  The part of its input patch (the tile and the halo of the depthwise windows) that lies in the image goes
// to LDS once, straight from global memory.  Each wavefront then takes 16 hidden channels at a time, by itself:
//   expand     v_mfma_f32_16x16x4f32, 16 channels x 16 patch pixels, filter in registers (read in the MFMA's own order, two k-steps
//              an instruction: the executor uploads it so; four-byte loads took twice as long), into a slab of its own
//              [channel][pixel]; pixels outside the image are zeros, the depthwise padding;
//   depthwise  a lane has one channel, its nine filter values in registers, and a quarter of the squares: (3 + S)^2 reads serve
//              four windows of nine;
//   project    the 16 channels are four k-steps of the projection, all output channels x the tile, accumulated over the
//              wavefront's channels.
// There is no barrier between the patch and the end, where the wavefronts' sums meet in LDS.  Where the tiles are few the
// hidden channels are also cut over workgroups: partial sums through the handle's scratch, the last to arrive adds them in
// order and finishes the tile (igemm_f32_small.hip states what the hand-over rests on); nobody waits for anybody.
//
// What bounds it: at batch 1 the chain of one launch, which replaces three; with many tiles the fp32 matrix pipes, shared with
// the vector instructions, and LDS reads.  96 -> 576 -> 96 channels at 14x14, batch 1, 10.2 us, in cycles: patch and filters
// 4100, expansion 4000, depthwise 600, projection 1200, sums in LDS 2000, hand-over 5600 (2200 until the counter is back, the
// nine parts 3400), stores 1200.
//
// Measured against the three calls, whole MobileNetV2 in a replayed graph (us): batch 1 254 -> 190, 2 284 -> 208, 4 332 -> 259,
// 8 413 -> 342, 16 556 -> 473, 32 800 -> 648, 64 1334 -> 1105.  Blocks alone at batch 1: 16 -> 96 -> 24 at 112x112 stride 2 8.5,
// 24 -> 144 -> 24 at 56x56 9.3, 32 -> 192 -> 32 at 28x28 7.8, 64 -> 384 -> 64 at 14x14 9.2, 160 -> 960 -> 160 at 7x7 12.7.  Tiles of
// 64 pixels were slower than 32 at every batch (24 -> 144 -> 24, batch 64: 112 against 89).
//
// Sums run in another order than the three calls', and start at the bias that those add last.
#include "igemm_f32.h"
#include "dnnrt_exec.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace dnnrt {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *lds_ptr;

struct BlockF32Args {
  const float *X, *W1, *b1, *Wd, *bd, *W3, *b3, *Z;  // b1, bd, b3, Z may be null; Z is laid out like Y
  float *Y;
  int Cin, Ch, Cout, H, W, P, Q, ph, pw;
  int TH, TW, QW, squares, PH, PW;  // tile, its 2 x 2 squares across and in all, its patch
  int kc, groups, per_split, splits, mb;  // k-steps of the expansion; groups of 16 hidden channels, of a part; blocks of 16 output channels
  int tiles_w, tiles_hw, tiles, units;    // units: tiles x parts x ranges of output channels
  unsigned magic_tiles, magic_splits, magic_tiles_w, magic_tiles_hw, magic_qw;
  float lo1, hi1, lod, hid, lo, hi;
};

__device__ __forceinline__ float clamp_keeping_nan(float v, float lo, float hi) {
  v = v < lo ? lo : v;
  return v > hi ? hi : v;
}

// A barrier that waits for this wavefront's LDS accesses but not for its loads from global memory.
__device__ __forceinline__ void lds_barrier32() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// S: the depthwise stride.  KC: most k-steps of four input channels (0: no expansion, X holds the hidden channels).  MB: most
// blocks of 16 output channels.  NB: blocks of 16 output pixels.
// Floats between the patch's channels in LDS (8 modulo 32: every other row's 16 pixels, four of them, meet none of the 64 banks
// twice) and between those of a slab (4 modulo 16: nor do 16 channels of a pixel); patches that need more are not taken.
constexpr int block32_xs(int s, int nb) { return s == 1 ? 72 : nb == 1 ? 136 : 200; }
constexpr int block32_ss(int s, int nb) { return s == 1 ? (nb == 1 ? 52 : 84) : nb == 1 ? 100 : 164; }
constexpr int block32_kg(int kc) { return kc <= 8 ? 2 : 8; }  // k-steps of a chunk
// Floats from the patch on that a workgroup's LDS holds at least: an expansion reads its chunks ahead through all of the template's k-steps, also
// where the block has fewer, and up to 15 pixels past a channel's end.  What lies there is read and not used.  (Reads that stop with the
// block's own steps took 191 us for a MobileNetV2 at batch 1 where these take 188.5.)
constexpr int block32_reach(int kc, int xs) { return kc > 0 ? 4 * kc * xs + 15 : 0; }
constexpr int block32_s2(int nb) { return nb == 1 ? 24 : 40; }  // between those of the depthwise results, as the patch's

template <int S, int KC, int MB, int NB>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(KC <= 8 ? 4 : 2))) void conv_f32_block_kernel(const BlockF32Args a, float *partials, unsigned *counters) {
#if __HIP_DEVICE_COMPILE__
  constexpr bool EXPAND = KC > 0;
  constexpr int XS = block32_xs(S, NB), SS = block32_ss(S, NB), S2 = block32_s2(NB);
  constexpr int KG = block32_kg(KC);        // the k-steps of an expansion are a multiple of this
  constexpr int WIN = 3 + S;                // rows and columns of input under a square
  constexpr int PAIRS = (MB * NB + 3) / 4;  // 16 x 16 blocks of the result a wavefront finishes, at most
  extern __shared__ __attribute__((aligned(1024))) float smem32[];
  // What the first loads need of the arguments, all at once: read where they are first used, each round is a fraction of a microsecond
  // (MobileNetV2 at batch 1 190.7 -> 188.4 us).
  asm volatile("" ::"s"(a.X), "s"(a.W1), "s"(a.Cin), "s"(a.H), "s"(a.W), "s"(a.ph), "s"(a.pw), "s"(a.TH), "s"(a.TW), "s"(a.PH), "s"(a.PW), "s"(a.kc), "s"(a.groups),
               "s"(a.per_split), "s"(a.splits), "s"(a.tiles_w), "s"(a.tiles_hw), "s"(a.tiles), "s"(a.units), "s"(a.magic_tiles), "s"(a.magic_splits),
               "s"(a.magic_tiles_w), "s"(a.magic_tiles_hw), "s"((int)blockDim.x));
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, l4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = (int)(blockDim.x >> 6);

  // neighbouring tiles of one range of hidden channels on one XCD: they share filters and halos in its L2
  const int unit = xcd_tile((int)blockIdx.x, a.units);
  if (unit < 0) return;
  const int us = div_magic(unit, a.tiles, a.magic_tiles), tile = unit - us * a.tiles;
  const int range = div_magic(us, a.splits, a.magic_splits), split = us - range * a.splits;
  const int n = div_magic(tile, a.tiles_hw, a.magic_tiles_hw), tr = tile - n * a.tiles_hw;
  const int ty = div_magic(tr, a.tiles_w, a.magic_tiles_w);
  const int p0 = ty * a.TH, q0 = (tr - ty * a.tiles_w) * a.TW;
  const int h0 = p0 * S - a.ph, w0 = q0 * S - a.pw;
  // the patch's part in the image: RH x RW pixels from (r0, c0) of the patch on
  const int r0 = max(0, -h0), c0 = max(0, -w0);
  const int RH = min(a.PH, a.H - h0) - r0, RW = min(a.PW, a.W - w0) - c0;
  constexpr bool ROWS = KC >= 24;
  const int row = ROWS ? (RW + 3) & ~3 : RW, NP = RH * row;  // in LDS, where ROWS pads a row to a multiple of four
  const unsigned inv_row = (65536u + row - 1) / (unsigned)row;  // px / row = px * inv_row >> 16 for px < 1024
  auto row_of = [&](int px) { return (int)((unsigned)px * inv_row >> 16); };
  const int HW = a.H * a.W, m_first = range * MB, mb = min(MB, a.mb - m_first);

  constexpr unsigned OUT = 0x80000000u;
  constexpr int AGENT = 16;  // the cache policy of device-scope accesses (sc1)
  auto rsrc_of = [](const float *w, int n) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(w), 0, w ? 4 * n : 0, 0x00020000); };
  const auto w1_rsrc = rsrc_of(a.W1, a.Cin * a.Ch), wd_rsrc = rsrc_of(a.Wd, 9 * a.Ch), w3_rsrc = rsrc_of(a.W3, a.Ch * a.Cout);
  const auto b1_rsrc = rsrc_of(a.b1, a.Ch), bd_rsrc = rsrc_of(a.bd, a.Ch), b3_rsrc = rsrc_of(a.b3, a.Cout);
  const auto x_rsrc = rsrc_of(a.X + (int64_t)n * a.Cin * HW, a.Cin * HW);
  auto load = [](__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0)); };

  float *Xs = smem32, *mine = smem32 + (EXPAND ? 4 * a.kc * XS : 0) + wave * (16 * (SS + S2)), *res = mine + 16 * SS;

  // Filters and biases of a group of 16 hidden channels: each requested for the next group as soon as this one's are used up.
  // The 1x1 filters come in blocks of 16 rows and eight columns, this lane's column l16 at k 2 l4 and 2 l4 + 1: two k-steps.
  [[maybe_unused]] floatx2 wa[EXPAND ? KC / 2 : 1];
  [[maybe_unused]] floatx4 bias;
  float wd[9], bd;
  floatx2 wp[2][MB];
  auto load2 = [](__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) { return __builtin_bit_cast(floatx2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0)); };
  auto load4 = [](__amdgpu_buffer_rsrc_t r, unsigned voff) { return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, 0, 0)); };
  auto load_expand = [&](int g) {
    if constexpr (EXPAND) {
      int cin = a.Cin;
      asm volatile("" : "+s"(cin));  // nothing below is kept in scalar registers for the whole kernel
      const unsigned first = 64u * (unsigned)(g * cin);
#pragma unroll
      for (int k = 0; k < KC / 2; k++) wa[k] = load2(w1_rsrc, 8 * k < cin ? 8u * (unsigned)lane : OUT, 8 * k < cin ? first + 512u * (unsigned)k : 0u);
      bias = load4(b1_rsrc, 4u * (unsigned)(16 * g + 4 * l4));
    }
  };
  auto load_depthwise = [&](int g) {
    const unsigned at = 4u * (unsigned)(16 * g + l16);
#pragma unroll
    for (int t = 0; t < 9; t++) wd[t] = load(wd_rsrc, at, 4u * (unsigned)(t * a.Ch));
    bd = load(bd_rsrc, at, 0);
  };
  auto load_project = [&](int g) {
    int cout = a.Cout;
    asm volatile("" : "+s"(cout));
#pragma unroll
    for (int m = 0; m < MB; m++) {
      const int row0 = 16 * (m_first + m), in = min(16, cout - row0);  // rows past Cout are not stored
      const unsigned at = 8u * (unsigned)(l4 * in + l16), first = row0 < cout ? 4u * (unsigned)(row0 * a.Ch + 16 * g * in) : 0u;
#pragma unroll
      for (int k = 0; k < 2; k++) wp[k][m] = load2(w3_rsrc, at, first + 32u * (unsigned)(k * max(in, 0)));
    }
  };
  const int g_end = min(a.groups, (split + 1) * a.per_split);
  int g = split * a.per_split + wave;
  // The patch is requested first, then the first group's filters; where channels are many a lane has four pixels of a row.
  typedef std::conditional_t<ROWS, floatx4, float> patch_t;
  constexpr int V = ROWS ? 4 : 1, AHEAD = ROWS ? 6 : 10;
  const int across = ROWS ? row >> 2 : row, units = RH * across, all = EXPAND ? a.Cin * units : 0;
  const unsigned inv_units = ((1u << 22) + units - 1) / (unsigned)units, inv_across = ROWS ? (65536u + across - 1) / (unsigned)across : inv_row;
  patch_t q[AHEAD];
  auto patch_unit = [&](int u, int &c, int &ur) { c = (int)((unsigned)u * inv_units >> 22); ur = u - c * units; };
  auto request = [&](int u0) {
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      int c, ur;
      patch_unit(min(u0 + i * 64 * G, all - 1), c, ur);
      const int r = (int)((unsigned)ur * inv_across >> 16), at = 4 * (c * HW + (h0 + r0 + r) * a.W + w0 + c0 + V * (ur - r * across));
      if constexpr (ROWS) q[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, at, 0, 0));
      else q[i] = load(x_rsrc, (unsigned)at, 0);
    }
  };
  auto settle = [&](int u0) {
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      int c, ur;
      patch_unit(min(u0 + i * 64 * G, all - 1), c, ur);
      *reinterpret_cast<patch_t *>(Xs + c * XS + V * ur) = q[i];
    }
  };
  if constexpr (EXPAND) request(tid);
  load_expand(min(g, a.groups - 1));
  load_depthwise(min(g, a.groups - 1));
  load_project(min(g, a.groups - 1));
  if constexpr (EXPAND) {
    settle(tid);
    for (int u0 = tid + AHEAD * 64 * G; u0 < all; u0 += AHEAD * 64 * G) {
      request(u0);
      settle(u0);
    }
    if constexpr (KG > 2)
      for (int u = a.Cin * XS + tid; u < 4 * a.kc * XS; u += 64 * G) Xs[u] = 0.f;  // what a last chunk has beside its channels
  }
  if (RH < a.PH || RW < a.PW)  // the depthwise padding, written once: expansions leave it as it is
    for (int u = lane; u < 4 * SS; u += 64) *reinterpret_cast<floatx4 *>(mine + 4 * u) = floatx4{0.f, 0.f, 0.f, 0.f};

  floatx4 acc[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[m][b] = floatx4{0.f, 0.f, 0.f, 0.f};
  lds_barrier32();

  for (; g < g_end; g += G) {
    const bool more = g + G < g_end;
    // ---- expand ---------------------------------------------------------------
    if constexpr (EXPAND) {
      // `blocks` of 16 pixels from p on
      auto expand = [&](int p, auto blocks_c) {
        constexpr int BLOCKS = decltype(blocks_c)::value;
        floatx4 e[BLOCKS];
#pragma unroll
        for (int u = 0; u < BLOCKS; u++) e[u] = bias;
        const float *xp = Xs + 2 * l4 * XS + p + l16;
        // a chunk's pixels are read while the chunk before is multiplied; what lies behind the last (block32_reach) is not used
        float x[2][KG][BLOCKS];
        auto read = [&](int k0, float (&to)[KG][BLOCKS]) {
#pragma unroll
          for (int k = 0; k < KG; k++)  // step k: channels 8 (k / 2) + 2 l4 + k % 2
#pragma unroll
            for (int u = 0; u < BLOCKS; u++) to[k][u] = xp[(8 * ((k0 + k) >> 1) + (k & 1)) * XS + 16 * u];
        };
        read(0, x[0]);
#pragma unroll
        for (int k0 = 0; k0 < KC; k0 += KG) {
          if (k0 + KG < KC) read(k0 + KG, x[(k0 / KG + 1) & 1]);
          if (k0 < a.kc)
#pragma unroll
            for (int k = 0; k < KG; k++)
#pragma unroll
              for (int u = 0; u < BLOCKS; u++) e[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[(k0 + k) >> 1][k & 1], x[(k0 / KG) & 1][k][u], e[u], 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < BLOCKS; u++) {
          const int px = p + 16 * u + l16, r = row_of(px);
          float *to = mine + 4 * l4 * SS + (r0 + r) * a.PW + c0 + px - r * row;
          if (px < NP && (!ROWS || px - r * row < RW))
#pragma unroll
            for (int i = 0; i < 4; i++) to[i * SS] = clamp_keeping_nan(e[u][i], a.lo1, a.hi1);
        }
      };
      int p = 0;
      for (; p + 16 < NP; p += 32) expand(p, std::integral_constant<int, 2>{});
      if (p < NP) expand(p, std::integral_constant<int, 1>{});
      if (more) load_expand(g + G);
    } else {
      for (int c64 = 0; c64 < NP; c64 += 64) {
        const int px = min(c64 + lane, NP - 1), r = row_of(px);
        const unsigned voff = 4u * (unsigned)((h0 + r0 + r) * a.W + w0 + c0 + px - r * row);
        float *to = mine + (r0 + r) * a.PW + c0 + px - r * row;
        float v[16];
#pragma unroll
        for (int c = 0; c < 16; c++) v[c] = load(x_rsrc, voff, 4u * (unsigned)((16 * g + c) * HW));
#pragma unroll
        for (int c = 0; c < 16; c++) to[c * SS] = v[c];
      }
    }
    // only this wavefront touches its slab, and its LDS accesses stay in order
    asm volatile("" ::: "memory");
    // ---- depthwise ------------------------------------------------------------
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int own = 4 * i + l4, sq = own < a.squares ? own : 0;  // squares past the tile repeat its first
      const int sy = div_magic(sq, a.QW, a.magic_qw), sx = sq - sy * a.QW;
      const float *win = mine + l16 * SS + 2 * S * (sy * a.PW + sx);
      floatx4 sum = {bd, bd, bd, bd};
#pragma unroll
      for (int r = 0; r < WIN; r++) {
        float h[WIN];
#pragma unroll
        for (int c = 0; c < WIN; c++) h[c] = win[r * a.PW + c];
#pragma unroll
        for (int o = 0; o < 4; o++) {
          const int t = r - (o >> 1) * S;
          if (t < 0 || t > 2) continue;
#pragma unroll
          for (int s = 0; s < 3; s++) sum[o] = fmaf(h[(o & 1) * S + s], wd[3 * t + s], sum[o]);
        }
      }
#pragma unroll
      for (int o = 0; o < 4; o++) sum[o] = clamp_keeping_nan(sum[o], a.lod, a.hid);
      *reinterpret_cast<floatx4 *>(res + l16 * S2 + 4 * own) = sum;
    }
    if (more) load_depthwise(g + G);
    asm volatile("" ::: "memory");
    // ---- project --------------------------------------------------------------
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float v = res[(8 * (k >> 1) + 2 * l4 + (k & 1)) * S2 + 16 * b + l16];
#pragma unroll
        for (int m = 0; m < MB; m++)
          if ((m & ~1) < mb) acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wp[k >> 1][m][k & 1], v, acc[m][b], 0, 0, 0);
      }
    if (more) load_project(g + G);
    asm volatile("" ::: "memory");
  }

  // ---- the blocks this wavefront finishes: pair i is block (m, b) of number wave + i G --------------------------
  const int pairs = mb * NB, PQ = a.P * a.Q;
  // the lane's first channel of four and its pixel in Y and Z, in bytes: past the end where there is none
  const auto z_rsrc = rsrc_of(a.Z ? a.Z + (int64_t)n * a.Cout * PQ : nullptr, a.Cout * PQ), y_rsrc = rsrc_of(a.Y + (int64_t)n * a.Cout * PQ, a.Cout * PQ);
  unsigned at[PAIRS];
  floatx4 zb[PAIRS], bb[PAIRS];
#pragma unroll
  for (int i = 0; i < PAIRS; i++) {
    const int pair = wave + i * G, m = pair / NB, b = pair - m * NB, co = 16 * (m_first + m) + 4 * l4;
    const int sq = 4 * b + (l16 >> 2), sy = div_magic(sq, a.QW, a.magic_qw), sx = sq - sy * a.QW;
    const int p = p0 + 2 * sy + (l16 >> 1 & 1), q = q0 + 2 * sx + (l16 & 1);
    at[i] = pair < pairs && sq < a.squares && p < a.P && q < a.Q && co < a.Cout ? 4u * (unsigned)(co * PQ + p * a.Q + q) : OUT;
    bb[i] = load4(b3_rsrc, 4u * (unsigned)co);
    if (a.Z)
#pragma unroll
      for (int j = 0; j < 4; j++) zb[i][j] = load(z_rsrc, at[i], 4u * (unsigned)(j * PQ));
  }
  lds_barrier32();  // nobody reads the patch or the slabs any more
  floatx4 *red = reinterpret_cast<floatx4 *>(smem32) + lane;  // [wavefront][pair][lane]
#pragma unroll
  for (int m = 0; m < MB; m++)
    if (m < mb)
#pragma unroll
      for (int b = 0; b < NB; b++) red[64 * (wave * pairs + m * NB + b)] = acc[m][b];
  lds_barrier32();
  floatx4 v[PAIRS];
#pragma unroll
  for (int i = 0; i < PAIRS; i++) {
    const int pair = wave + i * G;
    v[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (pair < pairs)
      for (int w = 0; w < G; w += 4) {  // G is four or eight
        floatx4 p[4];
#pragma unroll
        for (int u = 0; u < 4; u++) p[u] = red[64 * ((w + u) * pairs + pair)];
#pragma unroll
        for (int u = 0; u < 4; u++) v[i] += p[u];
      }
  }
  if (a.splits > 1) {
    const int slot = range * a.tiles + tile;
    constexpr int PART = MB * NB * 1024;  // bytes of a partial tile
    const auto part_rsrc = __builtin_amdgcn_make_buffer_rsrc(partials, 0, a.units * PART, 0x00020000);
    const unsigned mine_at = (unsigned)(slot * a.splits * PART + 16 * lane);
#pragma unroll
    for (int i = 0; i < PAIRS; i++) {
      const int pair = wave + i * G;
      if (pair < pairs) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uintx4, v[i]), part_rsrc, (int)mine_at, split * PART + 1024 * pair, AGENT);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();  // every wavefront's stores are where all XCDs agree, and the sums have been read
    volatile unsigned *arrived_s = reinterpret_cast<unsigned *>(smem32);
    if (tid == 0) *arrived_s = __hip_atomic_fetch_add(&counters[slot], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived_s != (unsigned)a.splits - 1) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (tid == 0) __hip_atomic_store(&counters[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < PAIRS; i++) v[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    constexpr int AT_ONCE = (KC <= 8 ? 16 : 32) / PAIRS < 16 ? (KC <= 8 ? 16 : 32) / PAIRS : 16;
    for (int y = 0; y < a.splits; y += AT_ONCE) {  // AT_ONCE parts in flight, added in order
      floatx4 o[AT_ONCE][PAIRS];
#pragma unroll
      for (int u = 0; u < AT_ONCE; u++)
#pragma unroll
        for (int i = 0; i < PAIRS; i++) {  // zeros behind the last, which cost no access
          const bool there = y + u < a.splits && wave + i * G < pairs;
          o[u][i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(part_rsrc, there ? (int)mine_at : (int)OUT, there ? (y + u) * PART + 1024 * (wave + i * G) : 0, AGENT));
        }
#pragma unroll
      for (int u = 0; u < AT_ONCE; u++)
#pragma unroll
        for (int i = 0; i < PAIRS; i++) v[i] += o[u][i];
    }
  }
#pragma unroll
  for (int i = 0; i < PAIRS; i++) {
    floatx4 y = v[i] + bb[i];
    if (a.Z) y += zb[i];
#pragma unroll
    for (int j = 0; j < 4; j++)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, clamp_keeping_nan(y[j], a.lo, a.hi)), y_rsrc, (int)at[i], 4 * j * PQ, 0);
  }
#endif
}

// ---- which problems, which cut -----------------------------------------------------
struct BlockF32Cut { int kc, mb, nb, G, lds, np; };  // the kernel's template arguments, wavefronts, bytes of LDS, pixels of a patch in LDS

static bool clamp_of(int64_t mode, float coef, float &lo, float &hi) {
  lo = mode == DNNRT_ACT_IDENTITY ? -__builtin_inff() : 0.f;
  hi = mode == DNNRT_ACT_CLIPPED_RELU ? coef : __builtin_inff();
  return mode == DNNRT_ACT_IDENTITY || mode == DNNRT_ACT_RELU || mode == DNNRT_ACT_CLIPPED_RELU;
}

constexpr int BLOCK32_LDS = 160 * 1024;

// Fills in `a` and `c` for a tile of 2 qh x 2 qw pixels in nb blocks of 16, G wavefronts and `splits` parts of the hidden
// channels; false where that cannot be.
static bool cut_block_f32(const dnnrtContext *ctx, const dnnrtExecBlock &k, int nb, int qw, int G, int splits, BlockF32Args &a, BlockF32Cut &c) {
  const int steps = (int)ceil_div(k.cin, 4);
  const int mall = (int)ceil_div(k.cout, 16);
  c.nb = nb; c.G = G;
  c.kc = !k.expand ? 0 : steps <= 8 && mall <= 2 ? 8 : steps <= 24 && mall <= 6 ? 24 : 40;
  c.mb = c.kc <= 8 ? 2 : c.kc == 24 ? 6 : 10;
  if (c.kc == 0 && mall > 2) return false;
  if (c.kc < 24 && nb != 2) return false;
  const int st = (int)k.stride, qh = std::min(4 * nb / qw, (int)(k.p + 1) / 2);
  if (qh < 1 || qw > 4 * nb) return false;
  a.Cin = (int)k.cin; a.Ch = (int)k.ch; a.Cout = (int)k.cout; a.H = (int)k.h; a.W = (int)k.w; a.P = (int)k.p; a.Q = (int)k.q;
  a.ph = (int)k.pad_h; a.pw = (int)k.pad_w;
  a.QW = qw; a.squares = qh * qw; a.TH = 2 * qh; a.TW = 2 * qw;
  a.PH = (a.TH - 1) * st + 3; a.PW = (a.TW - 1) * st + 3;
  a.kc = k.expand ? (int)ceil_div(steps, block32_kg(c.kc)) * block32_kg(c.kc) : 0;
  const int np = std::min(a.PH, a.H) * (c.kc >= 24 ? (std::min(a.PW, a.W) + 3) / 4 * 4 : std::min(a.PW, a.W));
  c.np = np;
  const int xs = block32_xs(st, nb), ss = block32_ss(st, nb);
  if (np > xs || a.PH * a.PW > ss) return false;
  a.groups = (int)ceil_div(k.ch, 16);
  a.per_split = (int)ceil_div(a.groups, splits);
  a.splits = (int)ceil_div(a.groups, a.per_split);
  if (a.splits != splits) return false;
  a.mb = mall;
  a.tiles_w = (int)ceil_div(a.Q, a.TW);
  a.tiles_hw = a.tiles_w * (int)ceil_div(a.P, a.TH);
  const int64_t tiles = k.n * a.tiles_hw, ranges = ceil_div(mall, c.mb), units = tiles * ranges * splits;
  if (units > (1 << 24)) return false;
  a.tiles = (int)tiles;
  a.units = (int)units;
  if (splits > 1 && (ctx->splitk_shared || tiles * ranges > ctx->splitk_max_tiles || units * c.mb * nb * 1024 > ctx->splitk_partial_bytes)) return false;
  c.lds = std::max({(4 * a.kc * xs + G * 16 * (ss + block32_s2(nb))) * 4, block32_reach(c.kc, xs) * 4, G * std::min(mall, c.mb) * nb * 1024});
  if (c.lds > BLOCK32_LDS) return false;
  a.magic_tiles = magic_of(a.tiles); a.magic_splits = magic_of(a.splits);
  a.magic_tiles_w = magic_of(a.tiles_w); a.magic_tiles_hw = magic_of(a.tiles_hw); a.magic_qw = magic_of(a.QW);
  return true;
}

// Estimated time of a cut in microseconds: fitted to 4300 cuts of MobileNetV2's twelve kinds of blocks at batch 1, 4, 16 and 64,
// 5 .. 140 us, within 10 % on the whole; the cut it picks takes 6 % more than the best of them on average.
static double block_f32_us(int num_cu, const dnnrtExecBlock &k, const BlockF32Args &a, const BlockF32Cut &c) {
  const int mb = std::min(a.mb, c.mb);
  const double group = (double)ceil_div(c.np, 16) * (20.5 * a.kc + (k.expand ? 288 : 173)) + 82.0 * c.nb * mb;  // cycles of a wavefront
  const double rounds = (double)ceil_div(a.per_split, c.G);
  const int per_cu = std::max(1, std::min(BLOCK32_LDS / c.lds, (c.kc <= 8 ? 16 : c.kc == 24 && c.nb == 1 ? 12 : 8) / c.G));
  const double at_once = std::min((double)per_cu, std::max(1.0, (double)a.units / num_cu)), waves = std::max(1.0, at_once * c.G / 4);  // of a compute unit; of a SIMD
  const double loads = (k.expand ? 1.43 * c.np * a.Cin / c.G : 0.0) + 12.3 * rounds * (4 * a.kc + 16 * c.mb);
  const double turn = rounds * group * std::max(waves, 1.4) + loads * at_once * c.G / 4 + 1790 + 790.0 * mb * c.nb;
  const double turns = std::max(1.0, (double)a.units / (at_once * num_cu));
  return 3.15 + turn * (turns + 0.57 * (std::ceil(turns) - turns)) / 2300 + (a.splits > 1 ? 1.7 : 0.0);
}

const dnnrtBlockCut *find_block_cut(const dnnrtContext *ctx, const int64_t (&sizes)[11]);  // conv_f16_block.hip
void keep_block_cut(const dnnrtContext *ctx, const int64_t (&sizes)[11], dnnrtBlockCut cut);

// `faster`: refuse what the separate calls do sooner.
static bool plan_block_f32(const dnnrtContext *ctx, const dnnrtExecBlock &k, bool faster, BlockF32Args &a, BlockF32Cut &c) {
  if (k.dtype != DNNRT_F32 || k.format != DNNRT_NCHW || k.r != 3 || k.s != 3 || (k.stride != 1 && k.stride != 2)) return false;
  if (k.cin < 1 || k.cin % 8 || k.ch < 1 || k.ch % 16 || k.cout < 1 || k.cout % 8 || k.ch > 4096 || k.cout > 4096 || (k.expand ? k.cin > 160 : k.cin != k.ch)) return false;
  // Every tile's patch must hold a row and a column of the image: tiles are two pixels or more, so a padding of up to two leaves one.
  if (k.n < 1 || k.h < 1 || k.w < 1 || k.pad_h < 0 || k.pad_h > 2 || k.pad_w < 0 || k.pad_w > 2) return false;
  if (k.h + 2 * k.pad_h < 3 || k.w + 2 * k.pad_w < 3 || k.p != (k.h + 2 * k.pad_h - 3) / k.stride + 1 || k.q != (k.w + 2 * k.pad_w - 3) / k.stride + 1) return false;
  const int64_t lim = 1ll << 28;  // elements of an image and of a filter: byte offsets below 2^31, what lies past an end included
  if (k.h * k.w > lim || k.p * k.q > lim || k.h * k.w * (k.cin + 16) > lim || k.p * k.q * (k.cout + 16) > lim || k.n > lim) return false;
  if ((k.expand && !clamp_of(k.act1, k.coef1, a.lo1, a.hi1)) || !clamp_of(k.actd, k.coefd, a.lod, a.hid) || !clamp_of(k.act, k.coef, a.lo, a.hi)) return false;
  const int64_t sizes[11] = {k.n, k.cin, k.h, k.w, k.ch, k.cout, k.stride, k.pad_h, k.pad_w, k.expand + 2 * k.dtype, ctx->splitk_partial_bytes};
  double best = 0;
  if (const dnnrtBlockCut *f = find_block_cut(ctx, sizes))
    if (cut_block_f32(ctx, k, f->nb, f->qw, f->waves, f->splits, a, c)) best = block_f32_us(ctx->num_cu, k, a, c);
  if (best == 0) {
    BlockF32Args t = a;
    BlockF32Cut u{};
    for (const int nb : {1, 2})
      for (int qw = 1; qw <= 4 * nb && (qw == 1 || 2 * (qw - 1) < k.q); qw++)
        for (const int G : {4, 8})
          for (int splits = 1; splits <= 32; splits++) {
            if (!cut_block_f32(ctx, k, nb, qw, G, splits, t, u)) continue;
            const double us = block_f32_us(ctx->num_cu, k, t, u);
            if (best == 0 || us < best) { best = us; a = t; c = u; }
            if (t.units >= 4 * ctx->num_cu) break;  // enough of them without cutting the channels further
          }
    if (best == 0) return false;
    keep_block_cut(ctx, sizes, dnnrtBlockCut{{}, c.nb, a.QW, c.G, a.splits});
  }
  // What the separate calls take, in microseconds; inside a network, whose other kernels had the caches, 15 % longer.
  const double in_px = (double)k.n * k.h * k.w, out_px = (double)k.n * k.p * k.q;
  const double us1 = k.expand ? std::max(4.7, 3 + in_px * (k.cin + k.ch) * 4 / 3.5e6 + 2 * in_px * k.cin * k.ch / 90e6) : 0;
  const double usd = std::max(3.5, 2 + (in_px + out_px) * k.ch * 4 / 3.5e6);
  const double us3 = std::max(4.7, 3 + out_px * (k.ch + k.cout) * 4 / 3.5e6 + 2 * out_px * k.ch * k.cout / 90e6);
  return !faster || best <= 1.15 * (us1 + usd + us3);
}

bool block_f32_applies(const dnnrtContext *ctx, const dnnrtExecBlock &k) {
  BlockF32Args a{};
  BlockF32Cut c{};
  return plan_block_f32(ctx, k, true, a, c);
}

template <int S, int KC, int MB, int NB>
static bool launch_one(const dnnrtContext *ctx, const BlockF32Args &a, const BlockF32Cut &c) {
  static LdsRaised raised;
  if (!raise_lds(raised, ctx->device, reinterpret_cast<const void *>(&conv_f32_block_kernel<S, KC, MB, NB>), BLOCK32_LDS)) {
    set_error("inverted residual block (fp32): cannot reserve %d bytes of LDS", BLOCK32_LDS);
    return false;
  }
  hipLaunchKernelGGL((conv_f32_block_kernel<S, KC, MB, NB>), dim3((unsigned)ceil_div(a.units, 8) * 8), dim3(64 * (unsigned)c.G), (size_t)c.lds, ctx->stream, a,
                     ctx->splitk_partials, ctx->splitk_counters);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("inverted residual block (fp32): launch failed: %s", hipGetErrorString(e)); return false; }
  return true;
}

template <int S>
static bool launch_stride(const dnnrtContext *ctx, const BlockF32Args &a, const BlockF32Cut &c) {
  switch (c.kc) {
    case 0: return launch_one<S, 0, 2, 2>(ctx, a, c);
    case 8: return launch_one<S, 8, 2, 2>(ctx, a, c);
    case 24: return c.nb == 1 ? launch_one<S, 24, 6, 1>(ctx, a, c) : launch_one<S, 24, 6, 2>(ctx, a, c);
    default: return c.nb == 1 ? launch_one<S, 40, 10, 1>(ctx, a, c) : launch_one<S, 40, 10, 2>(ctx, a, c);
  }
}

static void fill_operands(const dnnrtExecBlock &k, BlockF32Args &a) {
  auto f = [](const void *p) { return static_cast<const float *>(p); };
  a.X = f(k.x); a.W1 = f(k.w1); a.b1 = f(k.b1); a.Wd = f(k.wd); a.bd = f(k.bd); a.W3 = f(k.w3); a.b3 = f(k.b3); a.Z = f(k.z);
  a.Y = static_cast<float *>(k.y);
}

bool launch_block_f32(const dnnrtContext *ctx, const dnnrtExecBlock &k) {
  BlockF32Args a{};
  BlockF32Cut c{};
  if (!plan_block_f32(ctx, k, false, a, c)) { set_error("inverted residual block (fp32): not a shape this kernel takes"); return false; }
  fill_operands(k, a);
  return k.stride == 1 ? launch_stride<1>(ctx, a, c) : launch_stride<2>(ctx, a, c);
}

}  // namespace dnnrt

extern "C" void dnnrtExecBlockFilterF32(void *dst, const void *src, int64_t rows, int64_t cols) {
  const float *from = static_cast<const float *>(src);
  float *to = static_cast<float *>(dst);
  for (int64_t r0 = 0; r0 < rows; r0 += 16)
    for (int64_t c = 0; c < cols; c += 2)
      for (int64_t r = r0; r < rows && r < r0 + 16; r++)
        for (int64_t i = 0; i < 2; i++) *to++ = from[(c + i) * rows + r];
}
