// Row-major fp32 matrix product for transformer Linear layers:
//   D[M, N] = act(alpha * A[M, K] * B[K, N] + bias_col[n] + beta * Cin[m, n]),  A and B row-major.
//
// Tiles of 64x64; each of a workgroup's four wavefronts owns the whole tile for a quarter of the reduction, on
// v_mfma_f32_32x32x2f32.  Its operands go from global memory straight into a ring of two stages of 16 k that nobody else
// touches: no barrier, every operand read from LDS once (32 MFMAs per stage from 12 reads), nothing staged in registers.  The four sums meet
// in LDS, where each lane gets four neighbouring columns of four rows; bias and residual were requested before the first load.
//
// What bounds it: the matrix pipes (a stage is 2048 cycles of each SIMD's) and, with the one to a few tiles per compute unit of
// a few hundred rows, what stands around them: launch, first data, sums and epilogue 4 us, and the hand-over of the split
// reductions that let 24 tiles use 256 compute units.  The tiles left over after the last full round are split alone.
// M x K x N, us, before (64x64 tiles on eight wavefronts, chunks of 32 k staged through registers, a barrier per chunk) and now: 128 x
// 768 x 2304 12.7 -> 11.3, 768 x 3072 15.1 -> 13.8, 3072 x 768 16.0 -> 14.7; 384 rows 20.5 -> 16.6, 32.9 -> 24.4, 26.3 -> 22.7; 4096
// rows (the big-tile kernel of igemm_f32.hip before) 224 -> 133, 234 -> 174, 166 -> 158.
#include "igemm_f32.h"
#include "partials.h"

#include <type_traits>

namespace dnnrt {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));  // four words at any word address
typedef __attribute__((address_space(3))) void *lds_ptr;

[[maybe_unused]] constexpr unsigned F32W_OUT_OF_RANGE = 0x80000000u;  // above every num_records used here: reads as zeros
constexpr int F32W_BK = 16;                     // k of a stage
constexpr int F32W_STAGE = 2 * 64 * F32W_BK * 4;  // its bytes: 64 columns n and 64 rows m
constexpr int F32W_WAVE = 2 * F32W_STAGE;       // a wavefront's ring of two stages; later its 64x64 sums

// How a launch is cut: workgroups 0 .. units - 1 (a multiple of 8) are the split tiles' parts, the rest whole tiles.
struct Waves32Plan {
  int tiles_m, whole, rest, splits, units, stages_per_split;
  unsigned magic_tiles_m, magic_round;  // of tiles_m; of rest, rounded up to a multiple of 8
};

template <int N, int LGKM = 15>
__device__ __forceinline__ void f32w_wait() {  // s_waitcnt vmcnt(N) lgkmcnt(LGKM), 15: any; LDS accesses stay on their side of it
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (LGKM << 8));
  asm volatile("" ::: "memory");
}

__global__ __launch_bounds__(256, 2) void gemm_f32_waves_kernel(const IgemmArgs a, const Waves32Plan pl, float *partials, unsigned *counters) {
#if __HIP_DEVICE_COMPILE__
  constexpr int L = 8;  // loads of a stage
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  // ---- which tile, which stages: consecutive tiles (all rows m of one column range) on one XCD share B in its L2 ----
  const int stages = a.Kdim / F32W_BK;
  int tile, split = 0, s_beg = 0, s_end = stages;
  const int b = (int)blockIdx.x;
  const bool part = b < pl.units;
  if (part) {
    const int per_xcd = (pl.rest + 7) >> 3, w = div_magic(b, 8 * per_xcd, pl.magic_round), i = b - w * 8 * per_xcd;
    split = w;
    tile = (i & 7) * per_xcd + (i >> 3);
    if ((i >> 3) >= per_xcd || tile >= pl.rest) return;
    tile += pl.whole;
    s_beg = split * pl.stages_per_split;
    s_end = min(s_end, s_beg + pl.stages_per_split);
  } else {
    const int w = b - pl.units, per_xcd = (pl.whole + 7) >> 3;
    tile = (w & 7) * per_xcd + (w >> 3);
    if ((w >> 3) >= per_xcd || tile >= pl.whole) return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int tile_n = div_magic(tile, pl.tiles_m, pl.magic_tiles_m), tile_m = tile - tile_n * pl.tiles_m;
  const int n0 = tile_n * 64, m0 = tile_m * 64;
  char *ring = smem + wave * F32W_WAVE;

  // ---- this wavefront's stages ----------------------------------------------
  const int per_wave = (s_end - s_beg + 3) >> 2, my_beg = s_beg + wave * per_wave, nk = max(0, min(per_wave, s_end - my_beg));

  // What the lane finishes: columns out_n .. + 3 of the rows out_m + 16 o.  Bias and residual are requested first of all.
  const int out_m = m0 + (tid >> 4), out_n = n0 + 4 * (tid & 15), out_nc = min(out_n, a.Ncols - 4);
  floatx4 bias = {0.f, 0.f, 0.f, 0.f}, res[4];
  if (a.bias_col) bias = *reinterpret_cast<const float4u *>(a.bias_col + out_nc);
  if (a.Cin) {
#pragma unroll
    for (int o = 0; o < 4; o++) res[o] = *reinterpret_cast<const float4u *>(a.Cin + (int64_t)min(out_m + 16 * o, a.M - 1) * a.c_row_stride + out_nc);
  }

  // ---- loaders: byte offsets of this lane -----------------------------------
  // A: 64 bytes a row, 16-byte chunk c of row r at c ^ ((r >> 2) & 3), sixteen rows per instruction; B: as in memory, four k
  __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.A), 0, 4 * a.M * a.Kdim, 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.X), 0, 4 * a.Kdim * a.Ncols, 0x00020000);
  unsigned m_off[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int m = m0 + 16 * i + (lane >> 2);
    m_off[i] = m < a.M ? 4u * (unsigned)(m * a.Kdim + 4 * ((lane & 3) ^ ((lane >> 4) & 3))) : F32W_OUT_OF_RANGE;
  }
  const int b_n = n0 + 4 * (lane & 15);
  const unsigned n_off = b_n < a.Ncols ? 4u * (unsigned)((lane >> 4) * a.Ncols + b_n) : F32W_OUT_OF_RANGE;
  int l_k = F32W_BK * my_beg, l_slot = 0;
  auto issue_stage = [&]() {
    char *Ns = ring + l_slot, *Ms = Ns + 64 * F32W_BK * 4;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_ptr)(Ns + 1024 * i), 16, n_off, 4 * (l_k + 4 * i) * a.Ncols, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr)(Ms + 1024 * i), 16, m_off[i], 4 * l_k, 0, 0);
    }
    l_k += F32W_BK;
    l_slot ^= F32W_STAGE;
  };

  // ---- operand fetch: lane (l32, half) holds k 8 * half .. + 7; row i of block u is n 2 i + u, column i of block j is m 32 j + i ----
  floatx2 fn[2][8];
  floatx4 fm[2][2][2];
  const char *rd_n = ring + half * 2048 + 8 * l32, *rd_m = ring + 64 * F32W_BK * 4 + 64 * l32;
  const int chunk0 = 16 * ((2 * half) ^ ((l32 >> 2) & 3)), chunk1 = chunk0 ^ 16;
  int c_slot = 0;
  auto read_stage = [&](auto set_c) {
    constexpr int S = decltype(set_c)::value;
#pragma unroll
    for (int k = 0; k < 8; k++) fn[S][k] = *reinterpret_cast<const floatx2 *>(rd_n + c_slot + 256 * k);
#pragma unroll
    for (int j = 0; j < 2; j++) {
      fm[S][j][0] = *reinterpret_cast<const floatx4 *>(rd_m + c_slot + 2048 * j + chunk0);
      fm[S][j][1] = *reinterpret_cast<const floatx4 *>(rd_m + c_slot + 2048 * j + chunk1);
    }
    c_slot ^= F32W_STAGE;
  };
  floatx16 acc[2][2];
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[u][j][r] = 0.f;
  // The counted waits below assume that bias and residual are older than every ring load.
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  // ---- the reduction: nobody shares a ring, so there is no barrier ------------
  auto multiply = [&](auto set_c, auto q_c) {  // four of the stage's eight k of either half
    constexpr int S = decltype(set_c)::value, q = decltype(q_c)::value;
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[u][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fn[S][4 * q + e][u], fm[S][j][q][e], acc[u][j], 0, 0, 0);
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  auto step = [&](auto set_c, int ahead) {  // one stage, its operands in set S or on their way there; `ahead` follow it
    constexpr int S = decltype(set_c)::value;
    f32w_wait<63, 0>();  // its operands are here: its slot is free
    if (ahead >= 2) issue_stage();
    multiply(set_c, c0);
    __builtin_amdgcn_sched_barrier(0);
    if (ahead > 0) {
      if (ahead > 1) f32w_wait<L>();  // the next stage has landed, the one behind it may still be on its way
      else f32w_wait<0>();
      read_stage(std::integral_constant<int, 1 - S>{});
      __builtin_amdgcn_sched_barrier(0);
    }
    multiply(set_c, c1);
    __builtin_amdgcn_sched_barrier(0);
  };
  if (nk > 0) {
    issue_stage();
    if (nk > 1) {
      issue_stage();
      f32w_wait<L>();
    } else {
      f32w_wait<0>();
    }
    read_stage(c0);
    int ahead = nk - 1;
#pragma unroll 1
    for (; ahead > 0; ahead -= 2) {
      step(c0, ahead);
      step(c1, ahead - 1);
    }
    if (ahead == 0) step(c0, 0);
  }

  // ---- the four wavefronts' sums meet in LDS: [m][n], 16-byte chunk c of row m at c ^ (m & 15) ----
  // register r of block (u, j): n = 2 (8 (r / 4) + 4 half + r % 4) + u, m = 32 j + l32
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const floatx4 v = {acc[0][j][4 * g + 2 * p], acc[1][j][4 * g + 2 * p], acc[0][j][4 * g + 2 * p + 1], acc[1][j][4 * g + 2 * p + 1]};
        *reinterpret_cast<floatx4 *>(ring + (32 * j + l32) * 256 + 16 * ((4 * g + 2 * half + p) ^ (l32 & 15))) = v;
      }
  __syncthreads();
  floatx4 v[4];
#pragma unroll
  for (int o = 0; o < 4; o++) {
    const int m = (tid >> 4) + 16 * o;
    const char *at = smem + m * 256 + 16 * ((tid & 15) ^ (m & 15));
    v[o] = *reinterpret_cast<const floatx4 *>(at);
#pragma unroll
    for (int w = 1; w < 4; w++) v[o] += *reinterpret_cast<const floatx4 *>(at + w * F32W_WAVE);
  }

  // ---- a split reduction: the hand-over that igemm_f32_small.hip describes ----
  const int splits = pl.splits;
  if (part && splits > 1) {
    const int rt = tile - pl.whole;
    const __amdgpu_buffer_rsrc_t parts = part_rsrc(partials);
    const unsigned mine = 16u * (unsigned)tid, first_part = (unsigned)(rt * splits) * 16384u;
#pragma unroll
    for (int o = 0; o < 4; o++) part_store(parts, mine + 4096 * o, first_part + 16384u * (unsigned)split, v[o]);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    volatile unsigned *arrived = reinterpret_cast<unsigned *>(smem);
    if (tid == 0) *arrived = __hip_atomic_fetch_add(&counters[rt], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived != (unsigned)splits - 1) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (tid == 0) __hip_atomic_store(&counters[rt], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int o = 0; o < 4; o++) v[o] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int y0 = 0; y0 < splits; y0 += 4) {  // four parts requested at a time, added in split order
      part_floatx4 p[4][4];
#pragma unroll
      for (int y = 0; y < 4; y++)
#pragma unroll
        for (int o = 0; o < 4; o++)
          p[y][o] = part_load<part_floatx4>(parts, y0 + y < splits ? mine + 4096 * o : PART_NONE, first_part + 16384u * (unsigned)min(y0 + y, splits - 1));
#pragma unroll
      for (int y = 0; y < 4; y++)
#pragma unroll
        for (int o = 0; o < 4; o++) v[o] += p[y][o];
    }
  }

  // ---- epilogue ---------------------------------------------------------------
  if (out_n >= a.Ncols) return;
  auto finish = [&](auto mode_c) {
    constexpr int MODE = decltype(mode_c)::value;
#pragma unroll
    for (int o = 0; o < 4; o++) {
      floatx4 y;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float x = a.alpha * v[o][e] + bias[e];
        if (a.Cin) x += a.beta * res[o][e];
        y[e] = apply_act(x, MODE < 0 ? a.act : MODE, a.act_coef);
      }
      if (out_m + 16 * o < a.M) *reinterpret_cast<float4u *>(a.Y + (int64_t)(out_m + 16 * o) * a.y_row_stride + out_n) = y;
    }
  };
  if (a.act == DNNRT_ACT_IDENTITY) finish(std::integral_constant<int, DNNRT_ACT_IDENTITY>{});
  else if (a.act == ACT_GELU) finish(std::integral_constant<int, ACT_GELU>{});
  else finish(std::integral_constant<int, -1>{});
#endif
}

// Takes row-major products whose shape fits (returns launched = false otherwise).
bool launch_gemm_f32_waves(const dnnrtContext *ctx, const IgemmArgs &a, bool &launched) {
  launched = false;
  if (a.Z != 1 || a.b_kcontig || a.a_mcontig || a.bias || a.A2) return true;
  if (a.M < 1 || a.Ncols < 4 || a.Kdim % F32W_BK || a.Ncols % 4 || !aligned16(a.A) || !aligned16(a.X)) return true;
  const int64_t lim = (1ll << 31) - 4096;
  if (4 * (int64_t)a.M * a.Kdim > lim || 4 * (int64_t)a.Kdim * a.Ncols > lim) return true;
  // The operand-from-global kernels have the shorter chain while their 32x32 tiles are no more than one per compute unit over
  // 768 k or as much work as that: 300 x 768 x 768 9.0 us there, 10.6 here; 384 x 768 x 768 13.1 there, 11.3 here; 40 x 3072 x 768 10.4, 13.5;
  // 77 x 3072 x 768 14.5 either way.
  if (ceil_div(a.M, 32) * ceil_div(a.Ncols, 32) * a.Kdim <= (int64_t)ctx->num_cu * 768) return true;
  const int64_t tiles = ceil_div(a.M, 64) * ceil_div(a.Ncols, 64);
  if (tiles > (1 << 28)) return true;
  // Estimated microseconds: a stage of 16 k takes each of a workgroup's four wavefronts 0.95 (the matrix pipes: two workgroups on
  // a compute unit take twice that), everything around them 4, a split tile's hand-over 2.3 and 0.25 per part.  The tiles left
  // over after the last full round are split.
  const int stages = a.Kdim / F32W_BK;
  const int64_t rounds = tiles / ctx->num_cu, rest = tiles - rounds * ctx->num_cu;
  Waves32Plan pl{};
  double best = 0;
  for (int s = 1; s <= 16 && s <= stages; s++) {
    if (s > 1 && (ctx->splitk_shared || rest == 0 || rest > ctx->splitk_max_tiles || rest * s * 16384 > ctx->splitk_partial_bytes)) break;
    const int per = (int)ceil_div(stages, s);
    if (ceil_div(stages, per) != s) continue;  // no empty split: every arrival carries a partial tile
    const double load = (double)rounds * ceil_div(stages, 4) + (double)ceil_div(rest * s, ctx->num_cu) * ceil_div(per, 4);
    const double cost = 4.0 + 0.95 * load + (s > 1 ? 2.3 + 0.25 * s : 0);
    if (!pl.splits || cost < best) {
      best = cost;
      pl.splits = s;
      pl.rest = s > 1 ? (int)rest : 0;
      pl.whole = (int)tiles - pl.rest;
      pl.units = (int)ceil_div(pl.rest, 8) * 8 * s;
      pl.stages_per_split = per;
    }
  }
  if (!pl.splits) return true;
  pl.tiles_m = (int)ceil_div(a.M, 64);
  pl.magic_tiles_m = magic_of(pl.tiles_m);
  pl.magic_round = magic_of(pl.rest > 0 ? (int)ceil_div(pl.rest, 8) * 8 : 8);
  const unsigned grid = (unsigned)(pl.units + ceil_div(pl.whole, 8) * 8);
  hipLaunchKernelGGL(gemm_f32_waves_kernel, dim3(grid), dim3(256), 4 * F32W_WAVE, ctx->stream, a, pl, ctx->splitk_partials, ctx->splitk_counters);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("gemm_f32(waves): launch failed: %s", hipGetErrorString(e)); return false; }
  launched = true;
  return true;
}

}  // namespace dnnrt
