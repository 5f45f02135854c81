// fp32 3x3 convolution with stride 1 (filters C,R,S,K) by Winograd's minimal filtering F(2x2, 3x3) (S. Winograd, Arithmetic
// Complexity of Computations, 1980; A. Lavin, S. Gray, Fast Algorithms for Convolutional Neural Networks, 2015) on
// v_mfma_f32_32x32x2f32: 16 products per channel give four results of a filter instead of 36.
//
// A 2x2 tile of results needs a 4x4 patch d of its channel and becomes Y = At (sum over channels of (G g Gt) * (Bt d B)) A,
// the products element by element: for each of the 16 positions a matrix product [filter][channel] x [channel][tile].
// A workgroup has 64 filters and 32 tiles (128 pixels); wavefront i computes the four positions of row i, so that both
// transforms go one way across the wavefronts (each reads the patch and filter rows its own row needs) and one way inside
// a lane.  Nothing transformed is ever stored: raw filters and raw patches go from global memory straight into LDS
// (buffer_load ... lds, a ring of four stages of four channels, padding and edges are lanes whose offset reads zeros), and a
// lane turns what it reads into its MFMA operands.
//
// What bounds it: the matrix pipes and the vector instructions beside them, which on this chip take turns for fp32 (26 of
// them per eight MFMAs, 512 + 17 + 26 * 4.4 cycles).  512 workgroups of 64 stages, two per compute unit, take 94 us (205
// TFLOP/s of the direct form's operations, 157 being the chip's fp32 rate; 73 with nothing but the MFMAs left in).  Against the direct
// tiles of conv_f32_dma.hip, microseconds: 256 -> 512 channels at 56x56, two images, 134 -> 87; 1024 -> 324 at 38x38, three
// images, 273 -> 165; 64 -> 64 at 56x56, 32 images, 72 -> 49; 512 -> 512 at 7x7, 32 images, 80 -> 55.
//
// Precision: the transforms add four values of a patch and nine of a filter in fp32, and the sums run over C channels
// instead of 9 C products.  Relative error (2-norm) against 64-bit sums, the direct kernels' in brackets, over 64, 256 and
// 1024 channels: Gaussian filters, images after a ReLU 2.3e-7 (3.0e-7), 4.2e-7 (5.3e-7), 8.3e-7 (1.1e-6).  That holds for
// dense values; the transforms fill in zeros, and the direct sums of few products round less often.  A fifth of the
// activations non-zero: 1.05, 1.08 and 1.02 of the direct error, a twentieth 1.43, 1.32, 1.20.  Half the filter values
// zero: 1.00, 1.07, 1.01, nine tenths 1.61, 1.63, 1.52; that with a twentieth of the activations 2.46, 2.36, 2.27.  Per result the
// error is within (C + 27) 2^-24 of what magnitudes give in the same algorithm, which is the size of the 4x4 patch, not
// of the 3x3 window: next to values many orders of magnitude larger a result has no correct digits, and one whose products
// are all zero need not be zero.  The caller has the choice (DNNRT_CONV_ALGO_DIRECT); the executor makes it where a filter is
// mostly zero.
#include "igemm_f32.h"
#include "partials.h"

#include <type_traits>

namespace dnnrt {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));  // two words at any word address
typedef __attribute__((address_space(3))) void *lds_ptr;

[[maybe_unused]] constexpr unsigned W32_OUT_OF_RANGE = 0x80000000u;  // above every num_records used here: reads as zeros
constexpr int W32_BM = 64, W32_BT = 32;  // filters and 2x2 output tiles of a workgroup
constexpr int W32_BC = 4, W32_NS = 4;    // channels of a stage, stages of the ring
constexpr int W32_A_BYTES = 9 * W32_BC * W32_BM * 4;  // [pair of channels][tap][channel][filter]
constexpr int W32_STAGE = W32_A_BYTES + W32_BC * 16 * W32_BT * 4;  // [channel][row of the 4x4 patch][tile][column]
constexpr int W32_SMEM = W32_NS * W32_STAGE;
constexpr int W32_TILE = W32_BM * W32_BT * 4;  // results of a workgroup

// How a launch is cut: workgroups 0 .. units - 1 (a multiple of 8) are the split tiles' parts, the rest whole tiles.
struct Wino32Plan {
  int tiles_m, whole, rest, splits, units, stages, stages_per_split;
  int th, tw, n_tiles;  // 2x2 output tiles: per image down and across, all
  unsigned magic_tiles_m, magic_rest, magic_thw, magic_tw;
};

template <int FIRST, int LAST, class F>
__device__ __forceinline__ void w32_each(F f) {  // f(FIRST), .. f(LAST - 1), as constants
  if constexpr (FIRST < LAST) {
    f(std::integral_constant<int, FIRST>{});
    w32_each<FIRST + 1, LAST>(f);
  }
}

template <int AV>
__global__ __launch_bounds__(256, 2) void conv_f32_winograd_kernel(const IgemmArgs a, const Wino32Plan pl, float *partials, unsigned *counters) {
#if __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  // the arguments, all at once, as in conv_f32_dma.hip
  asm volatile("" ::"s"(pl.tiles_m), "s"(pl.whole), "s"(pl.rest), "s"(pl.splits), "s"(pl.units), "s"(pl.stages), "s"(pl.stages_per_split), "s"(pl.th), "s"(pl.tw),
               "s"(pl.n_tiles), "s"(pl.magic_tiles_m), "s"(pl.magic_rest), "s"(pl.magic_thw), "s"(pl.magic_tw), "s"(a.A), "s"(a.X), "s"(a.a_ld), "s"(a.M),
               "s"(a.Kdim), "s"(a.Ncols), "s"(a.H), "s"(a.W), "s"(a.P), "s"(a.Q), "s"(a.ph), "s"(a.pw), "s"(a.x_img_stride), "s"(a.magic_pq), "s"(a.bias));
  asm volatile("" ::"s"(a.Y), "s"(a.Cin), "s"(a.y_img_stride), "s"(a.y_row_stride), "s"(a.c_row_stride), "s"(a.act), "s"(a.act_coef), "s"(partials),
               "s"(counters));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;

  // ---- which tile, which stages -------------------------------------------
  int tile, split = 0, s_beg = 0, s_end = pl.stages;
  const int b = (int)blockIdx.x;
  const bool part = b < pl.units;
  if (part) {
    split = div_magic(b, pl.rest, pl.magic_rest);
    if (split >= pl.splits) return;
    tile = pl.whole + (b - split * pl.rest);
    s_beg = split * pl.stages_per_split;
    s_end = min(s_end, s_beg + pl.stages_per_split);
  } else {  // consecutive tiles (the filter rows of one range of pixels first) on one XCD: they share operands in its L2
    const int w = b - pl.units, per_xcd = (pl.whole + 7) >> 3;
    tile = (w & 7) * per_xcd + (w >> 3);
    if ((w >> 3) >= per_xcd || tile >= pl.whole) return;
  }
  const int tile_n = div_magic(tile, pl.tiles_m, pl.magic_tiles_m), tile_m = tile - tile_n * pl.tiles_m;
  const int m0 = tile_m * W32_BM;
  const int HW = a.H * a.W, C = a.Kdim / 9;

  const int thw = pl.th * pl.tw;
  struct Tile { bool ok; int img, ty, tx; };
  auto tile_at = [&](int i) -> Tile {  // 2x2 output tile i of this workgroup's 32
    const int t = tile_n * W32_BT + i;
    const bool in = t < pl.n_tiles;
    const int n = in ? div_magic(t, thw, pl.magic_thw) : 0, yx = in ? t - n * thw : 0, y = div_magic(yx, pl.tw, pl.magic_tw);
    return {in, n, y, yx - y * pl.tw};
  };

  // the bias of filter 16 wave + i is in lane i
  float bias_l = 0.f;
  if (a.bias) bias_l = a.bias[min(m0 + 16 * wave + (lane & 15), a.M - 1)];

  // ---- loaders: byte offsets of this lane ---------------------------------
  // A stage's filter rows lie pair by pair of channels, tap by tap, the two channels of a tap side by side, four rows to an
  // instruction (AV == 4): wavefront w loads rows 4 w .. + 3, 16 + 4 w .. + 3 and 32 + w.
  const int lda4 = 4 * (int)a.a_ld;
  __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.A), 0, (int)(a.Kdim * lda4), 0x00020000);
  const int a_m = m0 + (AV == 4 ? 4 * (lane & 15) : lane);
  auto filter_row = [](int i) { const int pair = i >= 18 ? 1 : 0, j = i - 18 * pair; return 9 * (2 * pair + (j & 1)) + (j >> 1); };
  [[maybe_unused]] unsigned a_v[3];
#pragma unroll
  for (int n = 0; n < 3; n++) {
    const int i = AV != 4 ? 0 : n < 2 ? 16 * n + 4 * wave + (lane >> 4) : 32 + wave;
    a_v[n] = a_m < a.M ? (unsigned)((AV == 4 ? filter_row(i) * lda4 : 0) + 4 * a_m) : W32_OUT_OF_RANGE;
  }
  // The 4x4 patches: four columns by 16 tiles of a row per instruction; wavefront w loads channel w's.
  __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(a.X), 0, (int)(4 * div_magic(a.Ncols, a.P * a.Q, a.magic_pq) * a.x_img_stride), 0x00020000);
  unsigned b_v[8];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const Tile t = tile_at(16 * h + (lane >> 2));
    const int iw = 2 * t.tx - a.pw + (lane & 3);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int ih = 2 * t.ty - a.ph + r;
      const bool in = t.ok && (unsigned)ih < (unsigned)a.H && (unsigned)iw < (unsigned)a.W;
      b_v[2 * r + h] = in ? 4u * (unsigned)(t.img * (int)a.x_img_stride + ih * a.W + iw) : W32_OUT_OF_RANGE;
    }
  }
  // The loads of a stage, one by one: the filter's first, then the patches'.
  constexpr int LA = AV == 4 ? 3 : 9, L = LA + 8;
  auto issue_load = [&](int stage, auto n_c) {
    constexpr int n = decltype(n_c)::value;
    char *As = smem + (stage & (W32_NS - 1)) * W32_STAGE;
    if constexpr (n < LA && AV == 4) {
      const int k0 = 9 * W32_BC * stage * lda4;
      if (n < 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr)(As + 4096 * n + 1024 * wave), 16, a_v[n], k0, 0, 0);
      else if (lane < 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr)(As + 8192 + 256 * wave), 16, a_v[2], k0, 0, 0);
    } else if constexpr (n < LA) {
      const int i = 9 * wave + n;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr)(As + 256 * i), 4, a_v[0], (9 * W32_BC * stage + filter_row(i)) * lda4, 0, 0);
    } else {
      char *Bs = As + W32_A_BYTES + wave * (16 * W32_BT * 4);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, (lds_ptr)(Bs + 256 * (n - LA)), 4, b_v[n - LA], 4 * HW * (stage * W32_BC + wave), 0, 0);
    }
  };
  // loads FIRST .. LAST - 1 of a stage
  auto issue_loads = [&](int stage, auto first_c, auto last_c) {
    constexpr int FIRST = decltype(first_c)::value, LAST = decltype(last_c)::value;
    w32_each<FIRST, LAST>([&](auto n_c) { issue_load(stage, n_c); });
  };

  // ---- the reduction -------------------------------------------------------
  // Wavefront i owns row i of the 4x4 transformed positions.  Of a channel it needs two rows of the patch,
  // x_i = d[ra] + sx d[rb], and of the filter g_i = g[0], (g[0] + g[2]) + g[1], (g[0] + g[2]) - g[1] or g[2]: the halves that
  // belong to the two in the middle, of rows as of columns, are applied to the sums (a power of two: the same bits).
  const int ra = wave == 2 ? 2 : wave == 0 ? 0 : 1, rb = wave == 2 ? 1 : wave == 3 ? 3 : 2;
  const float sx = wave == 1 ? 1.f : -1.f;
  const int g_base = wave == 3 ? 6 : 0;
  const float f1 = wave == 1 ? 1.f : wave == 2 ? -1.f : 0.f, f2 = wave == 1 || wave == 2 ? 1.f : 0.f;
  floatx16 acc[4][2];  // [column of the position][block]: row i of block u is filter 2 i + u
#pragma unroll
  for (int p = 0; p < 4; p++)
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[p][u][r] = 0.f;
  const char *rd_a = smem + half * 256 + 8 * l32;
  const char *rd_x = smem + W32_A_BYTES + half * (16 * W32_BT * 4) + 16 * l32;
  // A pair of channels is eight MFMAs, a stage two pairs.  An fp32 MFMA shares its multipliers with the vector instructions:
  // they run before or behind it, never under it (measured: 64 cycles per MFMA, 4.4 more per vector instruction and 17 per
  // change from the one to the other, with one wavefront on the SIMD as with two).  So a pair's operands are computed in one
  // go, behind the MFMAs of the pair before; what they are computed from is read a pair earlier, under its MFMAs.
  floatx2 g[2][9];
  floatx4 da[2], db[2];
  float U[4][2], V[4];
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  auto read_filter = [&](int at, auto pair_c) {  // channels 2 * pair + half of the stage at `at`
    constexpr int pair = decltype(pair_c)::value;
#pragma unroll
    for (int k = 0; k < 9; k++) {
      const int row = k < 3 ? g_base + k : k;
      g[pair][k] = *reinterpret_cast<const floatx2 *>(rd_a + at + (pair * 9 + row) * 512);
    }
  };
  auto read_patch = [&](int at, auto pair_c) {
    constexpr int pair = decltype(pair_c)::value;
    da[pair] = *reinterpret_cast<const floatx4 *>(rd_x + at + (pair * 8 + ra) * (4 * W32_BT * 4));
    db[pair] = *reinterpret_cast<const floatx4 *>(rd_x + at + (pair * 8 + rb) * (4 * W32_BT * 4));
  };
  auto transform = [&](auto pair_c) {
    constexpr int pair = decltype(pair_c)::value;
#pragma unroll
    for (int u = 0; u < 2; u++) {
      float h[3];
#pragma unroll
      for (int s = 0; s < 3; s++) h[s] = fmaf(f1, g[pair][3 + s][u], fmaf(f2, g[pair][6 + s][u], g[pair][s][u]));
      const float e = h[0] + h[2];
      U[0][u] = h[0];
      U[1][u] = e + h[1];
      U[2][u] = e - h[1];
      U[3][u] = h[2];
    }
    float x[4];
#pragma unroll
    for (int s = 0; s < 4; s++) x[s] = fmaf(sx, db[pair][s], da[pair][s]);
    V[0] = x[0] - x[2];
    V[1] = x[1] + x[2];
    V[2] = x[2] - x[1];
    V[3] = x[1] - x[3];
  };
  // This wavefront's part of the oldest stage in flight has landed, BEHIND younger ones may still be on their way; behind
  // the barrier that holds for all four wavefronts, and so does that they have read all of the stage before it.
  auto stage_ready = [&](auto behind_c) {
    constexpr int N = decltype(behind_c)::value * L;
    static_assert(N < 64, "vmcnt is a 6-bit counter");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));  // vmcnt(N) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#define PIN() __builtin_amdgcn_sched_barrier(0)
#define W32_MFMA(K) acc[(K) >> 1][(K) & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(U[(K) >> 1][(K) & 1], V[(K) >> 1], acc[(K) >> 1][(K) & 1], 0, 0, 0)
#define W32_LOADS(FROM, TO) if constexpr (AHEAD >= W32_NS) issue_loads(st + W32_NS, std::integral_constant<int, L * (FROM) / 12>{}, std::integral_constant<int, L * (TO) / 12>{})
  // AHEAD: stages that follow this one, W32_NS standing for so many or more.
  auto stage_body = [&](int st, auto ahead_c) {
    constexpr int AHEAD = decltype(ahead_c)::value;
    const int there = ((st + 1) & (W32_NS - 1)) * W32_STAGE;
    auto pair_body = [&](auto pair_c, auto other_c) {
      constexpr int pair = decltype(pair_c)::value;
      constexpr bool NEXT = pair < 1 || AHEAD > 0, READ = AHEAD > 0;  // a pair follows; one follows that one
      W32_MFMA(0);
      if constexpr (READ) read_filter(there, pair_c);
      PIN();
      W32_MFMA(1);
      if constexpr (READ) read_patch(there, pair_c);
      PIN();
      W32_MFMA(2);
      W32_LOADS(6 * pair, 6 * pair + 1);
      PIN();
      W32_MFMA(3);
      W32_LOADS(6 * pair + 1, 6 * pair + 2);
      PIN();
      W32_MFMA(4);
      W32_LOADS(6 * pair + 2, 6 * pair + 3);
      PIN();
      W32_MFMA(5);
      W32_LOADS(6 * pair + 3, 6 * pair + 4);
      PIN();
      W32_MFMA(6);
      W32_LOADS(6 * pair + 4, 6 * pair + 6);
      PIN();
      W32_MFMA(7);
      PIN();
      if constexpr (NEXT) transform(other_c);
      PIN();
    };
    if constexpr (AHEAD > 0) stage_ready(std::integral_constant<int, (AHEAD < W32_NS ? AHEAD : W32_NS - 1) - 1>{});
    PIN();
    pair_body(c0, c1);
    pair_body(c1, c0);
  };
  const int stages = s_end - s_beg;
#pragma unroll
  for (int i = 0; i < W32_NS; i++)
    if (i < stages) issue_loads(s_beg + i, c0, std::integral_constant<int, L>{});
  if (stages >= 4) stage_ready(std::integral_constant<int, 3>{});
  else if (stages == 3) stage_ready(std::integral_constant<int, 2>{});
  else if (stages == 2) stage_ready(c1);
  else stage_ready(c0);
  {
    const int at = (s_beg & (W32_NS - 1)) * W32_STAGE;
    read_filter(at, c0);
    read_patch(at, c0);
    read_filter(at, c1);
    read_patch(at, c1);
    transform(c0);
    PIN();
  }
  int st = s_beg;
  for (; st < s_end - 4; st++) stage_body(st, std::integral_constant<int, 4>{});
  if (stages > 3) stage_body(s_end - 4, std::integral_constant<int, 3>{});
  if (stages > 2) stage_body(s_end - 3, std::integral_constant<int, 2>{});
  if (stages > 1) stage_body(s_end - 2, c1);
  stage_body(s_end - 1, c0);
#undef W32_LOADS
#undef W32_MFMA
#undef PIN
  __syncthreads();  // nobody reads the operand stages any more

  // ---- back from the transformed positions: columns here, rows through LDS ----
  // [wavefront][filter 64][tile 32][2 columns]
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int row = 2 * (8 * (r >> 2) + 4 * half + (r & 3)) + u;
      const floatx2 v = {fmaf(0.5f, acc[1][u][r] + acc[2][u][r], acc[0][u][r]), fmaf(0.5f, acc[1][u][r] - acc[2][u][r], -acc[3][u][r])};
      *reinterpret_cast<floatx2 *>(smem + wave * (W32_TILE * 2) + (row * W32_BT + l32) * 8) = v;
    }
  __syncthreads();
  // This wavefront finishes filters 16 wave .. + 15; half the lanes the tiles' first rows, half the second.
  float v[16][2];
  {
    const char *rd = smem + half * (W32_TILE * 2) + (16 * wave * W32_BT + l32) * 8;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const floatx2 p = *reinterpret_cast<const floatx2 *>(rd + i * W32_BT * 8), q = *reinterpret_cast<const floatx2 *>(rd + W32_TILE * 2 + i * W32_BT * 8),
                    r = *reinterpret_cast<const floatx2 *>(rd + W32_TILE * 4 + i * W32_BT * 8);
#pragma unroll
      for (int j = 0; j < 2; j++) v[i][j] = fmaf(0.5f, half ? p[j] - q[j] : q[j] + r[j], half ? -r[j] : p[j]);
    }
  }

  // ---- a split tile: the hand-over of the other fp32 kernels (igemm_f32_small.hip states what it rests on) ----
  if (part && pl.splits > 1) {
    const int rt = tile - pl.whole;
    const __amdgpu_buffer_rsrc_t parts = part_rsrc(partials);
    const unsigned mine = 16u * (unsigned)tid, first_part = (unsigned)(rt * pl.splits) * (4u * W32_TILE);  // [two filters][thread]
#pragma unroll
    for (int i = 0; i < 16; i += 2)
      part_store(parts, mine + 2048 * i, first_part + (unsigned)split * (4u * W32_TILE), part_floatx4{v[i][0], v[i][1], v[i + 1][0], v[i + 1][1]});
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    volatile unsigned *arrived_s = reinterpret_cast<unsigned *>(smem);
    if (tid == 0) *arrived_s = __hip_atomic_fetch_add(&counters[rt], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived_s != (unsigned)pl.splits - 1) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (tid == 0) __hip_atomic_store(&counters[rt], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < 16; i++) v[i][0] = v[i][1] = 0.f;
    for (int y = 0; y < pl.splits; y += 4) {  // four partial tiles in flight, added in split order
      part_floatx4 p[4][8];
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int i = 0; i < 8; i++)
          p[u][i] = part_load<part_floatx4>(parts, y + u < pl.splits ? mine + 4096 * i : PART_NONE, first_part + (unsigned)min(y + u, pl.splits - 1) * (4u * W32_TILE));
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int i = 0; i < 32; i++) v[i >> 1][i & 1] += p[u][i >> 2][i & 3];
    }
  }

  // ---- epilogue: (acc + bias) + residual, activation ------------------------
  const Tile t = tile_at(l32);
  const bool ok = t.ok;
  const int img = t.img, p_out = 2 * t.ty + half, q_out = 2 * t.tx;
  const bool ok0 = ok && p_out < a.P, ok1 = ok0 && q_out + 1 < a.Q;
  const int64_t at = (int64_t)img * a.y_img_stride + (ok0 ? p_out * a.Q + q_out : 0);
  const int row0 = m0 + 16 * wave;
  const bool relu = a.act == DNNRT_ACT_RELU || a.act == DNNRT_ACT_CLIPPED_RELU;
  const float slope = a.act == DNNRT_ACT_LEAKY_RELU ? a.act_coef : 1.f, ceiling = a.act == DNNRT_ACT_CLIPPED_RELU ? a.act_coef : __builtin_inff();
  auto activate = [&](float x) {  // apply_act without a branch
    const float below = relu ? 0.f : slope * x;
    x = x < 0.f ? below : x;
    return x > ceiling ? ceiling : x;
  };
  // What is not finite here is computed again, tap by tap: differences of infinities, and sums that left fp32's range, are
  // none of the convolution's, and they spread over a tile.  The wavefront takes their pixels one by one, sixteen lanes to a
  // channel, a lane for each filter; finite results keep their bits, and once every sum is a NaN nothing more is read.
  // 1024 -> 324 channels at 38x38, three images, 184 us: with one NaN 198, an image of NaN 396, one infinity 1020.  (A lane
  // to a channel, 64 lines an instruction: 232, 833, 8870.  Every result of such a wavefront by its own lane: 28 ms each.)
  unsigned top = 0;
#pragma unroll
  for (int i = 0; i < 16; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) top = max(top, __builtin_bit_cast(unsigned, v[i][j]) & 0x7fffffffu);
  if (__builtin_expect(__any(top >= 0x7f800000u), 0)) {
    unsigned wrong[2] = {0, 0};  // bit i: filter row0 + i of pixel j
#pragma unroll
    for (int i = 0; i < 16; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        if (!(__builtin_fabsf(v[i][j]) < __builtin_inff()) && (j ? ok1 : ok0) && row0 + i < a.M) wrong[j] |= 1u << i;
    // in this wavefront's own rows of what it read above, behind the word of the hand-over: [pixel][filter][lane]
    float *there = reinterpret_cast<float *>(smem + W32_TILE * 2 + 16 * wave * W32_BT * 8) + lane;
    constexpr int PIXEL = W32_TILE * 2 / 4;
#pragma unroll
    for (int i = 0; i < 16; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) there[j * PIXEL + 64 * i] = v[i][j];
#pragma unroll 1
    for (int j = 0; j < 2; j++) {
      const unsigned mine = j ? wrong[1] : wrong[0];
#pragma unroll 1
      for (uint64_t pixels = __ballot(mine != 0); pixels; pixels &= pixels - 1) {
        const int l = __builtin_ctzll(pixels);
        const int ih0 = __builtin_amdgcn_readlane(p_out, l) - a.ph, iw0 = __builtin_amdgcn_readlane(q_out, l) + j - a.pw;
        const bool wanted = ((unsigned)__builtin_amdgcn_readlane((int)mine, l) >> (lane & 15)) & 1;
        const float *x = a.X + __builtin_amdgcn_readlane(img, l) * a.x_img_stride, *w = a.A + min(row0 + (lane & 15), a.M - 1);
        float s = 0.f, sum = 0.f;
#pragma unroll 1
        for (int c0 = 0; c0 < C; c0 += 8) {
          float xs[2][9], ws[2][9];
#pragma unroll
          for (int u = 0; u < 2; u++) {
            const int64_t c = min(c0 + 4 * u + (lane >> 4), C - 1);
#pragma unroll
            for (int k = 0; k < 9; k++) {
              xs[u][k] = x[c * HW + min(max(ih0 + k / 3, 0), a.H - 1) * a.W + min(max(iw0 + k % 3, 0), a.W - 1)];
              ws[u][k] = w[(c * 9 + k) * a.a_ld];
            }
          }
#pragma unroll
          for (int u = 0; u < 2; u++)
#pragma unroll
            for (int k = 0; k < 9; k++) {
              const bool in = (unsigned)(ih0 + k / 3) < (unsigned)a.H && (unsigned)(iw0 + k % 3) < (unsigned)a.W && c0 + 4 * u < C;
              s = in ? fmaf(ws[u][k], xs[u][k], s) : s;  // what is outside the image is no 0 to be multiplied
            }
          sum = s + __shfl_xor(s, 16);
          sum += __shfl_xor(sum, 32);
          if (__all(!wanted || __builtin_isnan(sum))) break;
        }
        for (unsigned rows = (unsigned)__builtin_amdgcn_readlane((int)mine, l); rows; rows &= rows - 1) {
          const int i = __builtin_ctz(rows);
          const float of_i = __shfl(sum, i);
          if (lane == l) there[j * PIXEL + 64 * i] = of_i;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 16; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) v[i][j] = there[j * PIXEL + 64 * i];
  }
  const bool full = row0 + 16 <= a.M, pairs = __all(!ok0 || ok1);  // every lane's two pixels are in the image
  float *__restrict__ Y = a.Y + at + (int64_t)row0 * a.y_row_stride;
  const float *__restrict__ Z = a.Cin ? a.Cin + at + (int64_t)row0 * a.c_row_stride : nullptr;
  auto finish = [&](auto pair_c) {
    constexpr bool PAIR = decltype(pair_c)::value;
    float z[16][2];
    if (Z) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const float *at_z = Z + (int64_t)min(i, a.M - 1 - row0) * a.c_row_stride;
        if constexpr (PAIR) {
          const float2u w = ok0 ? *reinterpret_cast<const float2u *>(at_z) : float2u{0.f, 0.f};
          z[i][0] = w[0]; z[i][1] = w[1];
        } else {
          z[i][0] = ok0 ? at_z[0] : 0.f;
          z[i][1] = ok1 ? at_z[1] : 0.f;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
      if (!full && row0 + i >= a.M) break;
      const float bias = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, bias_l), i));
      float x0 = v[i][0] + bias, x1 = v[i][1] + bias;
      if (Z) { x0 += z[i][0]; x1 += z[i][1]; }
      x0 = activate(x0);
      x1 = activate(x1);
      float *to = Y + (int64_t)i * a.y_row_stride;
      if constexpr (PAIR) {
        const float2u w = {x0, x1};
        if (ok0) *reinterpret_cast<float2u *>(to) = w;
      } else {
        if (ok0) to[0] = x0;
        if (ok1) to[1] = x1;
      }
    }
  };
  if (row0 >= a.M) return;
  if (pairs) finish(std::true_type{});
  else finish(std::false_type{});
#endif
}

bool launch_conv_f32_winograd(const dnnrtContext *ctx, const IgemmArgs &args, double at_most_us, bool &launched) {
  launched = false;
  IgemmArgs a = args;
  if (a.R != 3 || a.S != 3 || a.sh != 1 || a.sw != 1 || a.A2 || !a.a_mcontig || a.b_kcontig || a.Z != 1 || a.bias_col || a.alpha != 1.f ||
      (a.Cin && a.beta != 1.f) || a.act == ACT_GELU || a.Kdim % (9 * W32_BC))
    return true;
  const int PQ = a.P * a.Q, C = a.Kdim / 9;
  const int64_t images = a.Ncols / PQ, lim = (1ll << 31) - 4096;
  if (images * PQ != a.Ncols || a.x_img_stride < (int64_t)C * a.H * a.W || 4 * images * a.x_img_stride > lim || 4 * (int64_t)a.Kdim * a.a_ld > lim) return true;
  const bool av4 = a.M % 4 == 0 && a.a_ld % 4 == 0 && aligned16(a.A);
  Wino32Plan pl{};
  pl.th = (int)ceil_div(a.P, 2);
  pl.tw = (int)ceil_div(a.Q, 2);
  pl.n_tiles = (int)(images * pl.th * pl.tw);
  pl.tiles_m = (int)ceil_div(a.M, W32_BM);
  pl.stages = C / W32_BC;
  const int64_t tiles = pl.tiles_m * ceil_div(pl.n_tiles, W32_BT);
  if (tiles > (1 << 28)) return true;
  // Estimated time in microseconds: a stage takes a compute unit 0.62 whether one or two workgroups share it, a workgroup's
  // start and end 9 with the launch and 2.3 for every further one in a row, a split tile's hand-over 3.1 and 0.7 per part, a lone workgroup's stores to rows of odd length 1.4 (measured on layers
  // of 0.8 .. 26 GFLOP, 64 to 1320 tiles, within 12 %).  As in conv_f32_dma.hip the tiles left over after the last full round are split.
  const int64_t rounds = tiles / ctx->num_cu, rest = tiles - rounds * ctx->num_cu;
  double best = 0;
  for (int s = 1; s <= 16; s++) {
    if (s > 1 && (rest == 0 || ctx->splitk_shared || rest * s * W32_TILE * 4 > ctx->splitk_partial_bytes || rest > ctx->splitk_max_tiles)) break;
    const int per = (int)ceil_div(pl.stages, s);
    if (ceil_div(pl.stages, per) != s) continue;
    const int64_t parts = ceil_div(rest * s, ctx->num_cu);
    const double cost = 9.0 + 0.62 * ((double)rounds * pl.stages + (double)parts * per) + 2.3 * (double)(rounds + parts - 1) + (s > 1 ? 3.1 + 0.7 * s : 0.0) + (a.Q % 2 && rounds + parts == 1 ? 1.4 : 0.0);
    if (!pl.splits || cost < best) {
      best = cost;
      pl.splits = s;
      pl.rest = s > 1 ? (int)rest : 0;
      pl.whole = (int)tiles - pl.rest;
      pl.units = (int)(ceil_div((int64_t)pl.rest * s, 8) * 8);
      pl.stages_per_split = per;
    }
  }
  if (best > at_most_us) return true;
  pl.magic_tiles_m = magic_of(pl.tiles_m);
  pl.magic_rest = magic_of(pl.rest > 0 ? pl.rest : 1);
  pl.magic_thw = magic_of(pl.th * pl.tw);
  pl.magic_tw = magic_of(pl.tw);
  a.magic_pq = magic_of(PQ);
  launched = true;
  const unsigned grid = (unsigned)(pl.units + ceil_div(pl.whole, 8) * 8);
  const auto kernel = av4 ? conv_f32_winograd_kernel<4> : conv_f32_winograd_kernel<1>;
  static LdsRaised raised[2];
  if (!raise_lds(raised[av4], ctx->device, reinterpret_cast<const void *>(kernel), W32_SMEM)) {
    set_error("conv(fp32, winograd): cannot reserve %d bytes of LDS", W32_SMEM);
    return false;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), W32_SMEM, ctx->stream, a, pl, ctx->splitk_partials, ctx->splitk_counters);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("conv(fp32, winograd): launch failed: %s", hipGetErrorString(e)); return false; }
  return true;
}

}  // namespace dnnrt
