// Row-major fp32 matrix product for transformer Linear layers:
//   D[M, N] = act(alpha * A[M, K] * B[K, N] + bias_col[n] + beta * Cin[m, n]),  A and B row-major.
//
// Tiles of 64 columns and 64 or 32 rows; each of a workgroup's four wavefronts owns the whole tile for a quarter of the reduction,
// on v_mfma_f32_32x32x2f32.  Its operands go from global memory straight into a ring of two stages of 16 k that nobody
// else touches: no barrier, every operand read from LDS once (32 MFMAs per stage from 12 reads), nothing staged in registers.  The
// four sums meet in LDS, where each lane gets four neighbouring columns of some rows; bias and residual were requested behind the
// ring's first loads.
//
// What bounds it: the matrix pipes (a stage is 2048 or 1024 cycles of each SIMD's) and, with the one to a few tiles per compute
// unit of a few hundred rows, what stands around them: launch, first data, sums and epilogue 4 us, and the hand-over of the split
// reductions that let 24 tiles use 256 compute units: its last workgroup reads all parts by itself, 160 KB of ten at 128 x 3072 x
// 768, where 48 tiles of 32 rows need five parts of half the size.  The tiles left over after the last full round are split alone.
// M x K x N, us, tiles of 64 rows alone and with those of 32: 128 x 768 x 2304 11.8 -> 11.1 (no split any more), 768 x 3072 13.5 ->
// 11.4, 3072 x 768 15.2 -> 12.7; 160 rows 13.7 -> 11.2, 16.0 -> 11.4, 21.6 -> 14.3; 384 x 768 x 3072 25.2 -> 22.1; 512 x 768 x 768 13.0
// -> 11.0.  BERT fp32 at 128 tokens 790 -> 713.  4096 rows, 64 of them a tile: 133, 174 and 158.
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
constexpr int f32w_stage(int tm) { return (64 + 32 * tm) * F32W_BK * 4; }             // its bytes: 64 columns n and 32 tm rows m
// A wavefront's ring of two stages; later its sums.  With tiles of 32 rows a third stage costs where the weights come from HBM (340 MB in a
// fp32 BERT-base, 128 tokens: 627 us with two, 634 with three, 656 with four, 676 with five) and gives nothing where they do not.
constexpr int f32w_wave(int tm) { return 2 * f32w_stage(tm); }

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

// TM: blocks of 32 rows of a tile.  The arguments in front of the structs are in registers when a wavefront starts: all that the
// ring's first loads need, so that nothing waits for the rest, which comes 0.45 us later
// (a BERT-base over 128 tokens, 36 of its 88 launches here and 12 in the small 1x1 kernel, 702 -> 663 us).  They are in the structs too.
template <int TM>
__global__ __launch_bounds__(256, 2) void gemm_f32_waves_kernel(const float *A, const float *X, int M, int Kdim, int Ncols, int units, int rest, int whole,
                                                                int stages_per_split, int tiles_m, unsigned magic_round, unsigned magic_tiles_m,
                                                                const IgemmArgs args, const Waves32Plan plan, float *partials, unsigned *counters) {
#if __HIP_DEVICE_COMPILE__
  IgemmArgs a = args;
  a.A = A; a.X = X; a.M = M; a.Kdim = Kdim; a.Ncols = Ncols;
  const Waves32Plan pl = {tiles_m, whole, rest, 0, units, stages_per_split, magic_tiles_m, magic_round};
  constexpr int L = 4 + 2 * TM;  // loads of a stage
  constexpr int STAGE = f32w_stage(TM), WAVE = f32w_wave(TM), NS = WAVE / STAGE, TILE = 64 * 32 * TM;
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
  const int n0 = tile_n * 64, m0 = tile_m * 32 * TM;
  char *ring = smem + wave * WAVE;

  // ---- this wavefront's stages: every fourth, so that the four read neighbouring rows of B and the same lines of A's rows at a time (a quarter
  // each in a run: BERT-base over 128 tokens 627 -> 618 us) ----
  const int my_beg = s_beg + wave, nk = max(0, (s_end - my_beg + 3) >> 2);

  // ---- loaders: byte offsets of this lane -----------------------------------
  // A: 64 bytes a row, 16-byte chunk c of row r at c ^ ((r >> 2) & 3), sixteen rows per instruction; B: as in memory, four k
  __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.A), 0, 4 * a.M * a.Kdim, 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.X), 0, 4 * a.Kdim * a.Ncols, 0x00020000);
  unsigned m_off[2 * TM];
#pragma unroll
  for (int i = 0; i < 2 * TM; i++) {
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
      if (i < 2 * TM) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr)(Ms + 1024 * i), 16, m_off[i < 2 * TM ? i : 0], 4 * l_k, 0, 0);
    }
    l_k += 4 * F32W_BK;
    l_slot = l_slot + STAGE == WAVE ? 0 : l_slot + STAGE;
  };

  // ---- operand fetch: lane (l32, half) holds k 8 * half .. + 7; row i of block u is n 2 i + u, column i of block j is m 32 j + i ----
  floatx2 fn[2][8];
  floatx4 fm[2][TM][2];
  const char *rd_n = ring + half * 2048 + 8 * l32, *rd_m = ring + 64 * F32W_BK * 4 + 64 * l32;
  const int chunk0 = 16 * ((2 * half) ^ ((l32 >> 2) & 3)), chunk1 = chunk0 ^ 16;
  int c_slot = 0;
  auto read_stage = [&](auto set_c) {
    constexpr int S = decltype(set_c)::value;
#pragma unroll
    for (int k = 0; k < 8; k++) fn[S][k] = *reinterpret_cast<const floatx2 *>(rd_n + c_slot + 256 * k);
#pragma unroll
    for (int j = 0; j < TM; j++) {
      fm[S][j][0] = *reinterpret_cast<const floatx4 *>(rd_m + c_slot + 2048 * j + chunk0);
      fm[S][j][1] = *reinterpret_cast<const floatx4 *>(rd_m + c_slot + 2048 * j + chunk1);
    }
    c_slot = c_slot + STAGE == WAVE ? 0 : c_slot + STAGE;
  };
  // With half as many rows there is room for four sums of a quarter of the length: the precision that the larger tiles' split
  // reductions gave (128 x 768 x 2304, 2-norm against 64 bits: 1.5e-7 with one sum, 1.1e-7 with two, 0.86e-7 with four; 0.95e-7 in
  // three parts of the larger tiles).
  constexpr int SUMS = TM == 1 ? 4 : 1;
  floatx16 acc[2][TM], more[SUMS > 1 ? SUMS - 1 : 1][2][TM];
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int j = 0; j < TM; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        acc[u][j][r] = 0.f;
#pragma unroll
        for (int i = 0; i < SUMS - 1; i++) more[i][u][j][r] = 0.f;
      }
#pragma unroll
  for (int i = 0; i < NS; i++)
    if (i < nk) issue_stage();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // The other arguments, all at once: read where they are used, each is waited for there.
  int splits = plan.splits;
  asm volatile("" : "+s"(a.bias_col), "+s"(a.Cin), "+s"(a.c_row_stride), "+s"(a.Y), "+s"(a.y_row_stride), "+s"(a.alpha), "+s"(a.beta), "+s"(a.act),
               "+s"(a.act_coef), "+s"(splits), "+s"(partials), "+s"(counters));
  // What the lane finishes: columns out_n .. + 3 of the rows out_m + 16 o.  Bias and residual are requested behind the ring's
  // first loads; the counted waits below are for the loads of the ring alone, these make the first of them stricter.
  const int out_m = m0 + (tid >> 4), out_n = n0 + 4 * (tid & 15), out_nc = min(out_n, a.Ncols - 4);
  floatx4 bias = {0.f, 0.f, 0.f, 0.f}, res[2 * TM];
  if (a.bias_col) bias = *reinterpret_cast<const float4u *>(a.bias_col + out_nc);
  if (a.Cin) {
#pragma unroll
    for (int o = 0; o < 2 * TM; o++) res[o] = *reinterpret_cast<const float4u *>(a.Cin + (int64_t)min(out_m + 16 * o, a.M - 1) * a.c_row_stride + out_nc);
  }
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
        for (int j = 0; j < TM; j++) {
          constexpr int LAST = SUMS > 1 ? SUMS - 2 : 0;
          const int sum = SUMS > 1 ? 2 * q + (e & 1) : 0;
          floatx16 &to = sum ? more[min(sum - 1, LAST)][u][j] : acc[u][j];
          to = __builtin_amdgcn_mfma_f32_32x32x2f32(fn[S][4 * q + e][u], fm[S][j][q][e], to, 0, 0, 0);
        }
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  auto landed = [&](int behind) {  // the oldest stage in flight has landed, one behind it may still be on its way
    if (behind >= 1) f32w_wait<L>();
    else f32w_wait<0>();
  };
  auto step = [&](auto set_c, int ahead) {  // one stage, its operands in set S or on their way there; `ahead` follow it
    constexpr int S = decltype(set_c)::value;
    f32w_wait<63, 0>();  // its operands are here: its slot is free
    if (ahead >= NS) issue_stage();
    multiply(set_c, c0);
    __builtin_amdgcn_sched_barrier(0);
    if (ahead > 0) {
      landed(ahead - 1);
      read_stage(std::integral_constant<int, 1 - S>{});
      __builtin_amdgcn_sched_barrier(0);
    }
    multiply(set_c, c1);
    __builtin_amdgcn_sched_barrier(0);
  };
  if (nk > 0) {
    landed(nk - 1);
    read_stage(c0);
    int ahead = nk - 1;
#pragma unroll 1
    for (; ahead > 0; ahead -= 2) {
      step(c0, ahead);
      step(c1, ahead - 1);
    }
    if (ahead == 0) step(c0, 0);
  }

  if constexpr (SUMS > 1)
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int j = 0; j < TM; j++) acc[u][j] = (acc[u][j] + more[0][u][j]) + (more[1][u][j] + more[2][u][j]);
  // ---- the four wavefronts' sums meet in LDS: [m][n], 16-byte chunk c of row m at c ^ (m & 15) ----
  // register r of block (u, j): n = 2 (8 (r / 4) + 4 half + r % 4) + u, m = 32 j + l32
#pragma unroll
  for (int j = 0; j < TM; j++)
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const floatx4 v = {acc[0][j][4 * g + 2 * p], acc[1][j][4 * g + 2 * p], acc[0][j][4 * g + 2 * p + 1], acc[1][j][4 * g + 2 * p + 1]};
        *reinterpret_cast<floatx4 *>(ring + (32 * j + l32) * 256 + 16 * ((4 * g + 2 * half + p) ^ (l32 & 15))) = v;
      }
  __syncthreads();
  floatx4 v[2 * TM];
#pragma unroll
  for (int o = 0; o < 2 * TM; o++) {
    const int m = (tid >> 4) + 16 * o;
    const char *at = smem + m * 256 + 16 * ((tid & 15) ^ (m & 15));
    v[o] = *reinterpret_cast<const floatx4 *>(at);
#pragma unroll
    for (int w = 1; w < 4; w++) v[o] += *reinterpret_cast<const floatx4 *>(at + w * WAVE);
  }

  // ---- a split reduction: the hand-over that igemm_f32_small.hip describes ----
  if (part && splits > 1) {
    const int rt = tile - pl.whole;
    const __amdgpu_buffer_rsrc_t parts = part_rsrc(partials);
    const unsigned mine = 16u * (unsigned)tid, first_part = (unsigned)(rt * splits) * (4u * TILE);
#pragma unroll
    for (int o = 0; o < 2 * TM; o++) part_store(parts, mine + 4096 * o, first_part + 4u * TILE * (unsigned)split, v[o]);
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
    for (int o = 0; o < 2 * TM; o++) v[o] = floatx4{0.f, 0.f, 0.f, 0.f};
    constexpr int AT_ONCE = 8 / TM;
    for (int y0 = 0; y0 < splits; y0 += AT_ONCE) {  // so many parts requested at a time, added in split order
      part_floatx4 p[AT_ONCE][2 * TM];
#pragma unroll
      for (int y = 0; y < AT_ONCE; y++)
#pragma unroll
        for (int o = 0; o < 2 * TM; o++)
          p[y][o] = part_load<part_floatx4>(parts, y0 + y < splits ? mine + 4096 * o : PART_NONE, first_part + 4u * TILE * (unsigned)min(y0 + y, splits - 1));
#pragma unroll
      for (int y = 0; y < AT_ONCE; y++)
#pragma unroll
        for (int o = 0; o < 2 * TM; o++) v[o] += p[y][o];
    }
  }

  // ---- epilogue ---------------------------------------------------------------
  if (out_n >= a.Ncols) return;
  auto finish = [&](auto mode_c) {
    constexpr int MODE = decltype(mode_c)::value;
#pragma unroll
    for (int o = 0; o < 2 * TM; o++) {
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
  // Estimated microseconds: a stage of 16 k takes each of a workgroup's four wavefronts 0.95, with tiles of 32 rows 0.52 (the matrix
  // pipes: two workgroups on a compute unit take twice that), everything around them 4 and, with 32 rows, 1 more for every further
  // workgroup that a compute unit takes, a split tile's hand-over 2.3 and 0.25 per part (0.125).  The tiles left over after the last full
  // round are split.
  const int stages = a.Kdim / F32W_BK;
  Waves32Plan pl{};
  double best = 0;
  int tm = 2;
  for (int t = 2; t >= 1; t--) {
    const int64_t tiles = ceil_div(a.M, 32 * t) * ceil_div(a.Ncols, 64);
    if (tiles > (1 << 28)) return true;
    const int64_t rounds = tiles / ctx->num_cu, rest = tiles - rounds * ctx->num_cu;
    for (int s = 1; s <= 16 && s <= stages; s++) {
      if (s > 1 && (ctx->splitk_shared || rest == 0 || rest > ctx->splitk_max_tiles || rest * s * 8192 * t > ctx->splitk_partial_bytes)) break;
      const int per = (int)ceil_div(stages, s);
      if (ceil_div(stages, per) != s) continue;  // no empty split: every arrival carries a partial tile
      const int64_t parts = ceil_div(ceil_div(rest, 8) * s, ceil_div(ctx->num_cu, 8));  // on the busiest compute unit: tiles go to the XCDs
      const double load = (double)rounds * ceil_div(stages, 4) + (double)parts * ceil_div(per, 4);
      const double cost = 4.0 + (t == 2 ? 0.95 : 0.52) * load + (t == 1 ? 1.0 * (double)(rounds + parts - 1) : 0.0) + (s > 1 ? 2.3 + 0.125 * t * s : 0);
      if (!pl.splits || cost < best) {
        best = cost;
        tm = t;
        pl.splits = s;
        pl.rest = s > 1 ? (int)rest : 0;
        pl.whole = (int)tiles - pl.rest;
        pl.units = (int)ceil_div(pl.rest, 8) * 8 * s;
        pl.stages_per_split = per;
      }
    }
  }
  if (!pl.splits) return true;
  pl.tiles_m = (int)ceil_div(a.M, 32 * tm);
  pl.magic_tiles_m = magic_of(pl.tiles_m);
  pl.magic_round = magic_of(pl.rest > 0 ? (int)ceil_div(pl.rest, 8) * 8 : 8);
  const unsigned grid = (unsigned)(pl.units + ceil_div(pl.whole, 8) * 8);
  const auto kernel = tm == 2 ? gemm_f32_waves_kernel<2> : gemm_f32_waves_kernel<1>;
  const int lds = 4 * f32w_wave(tm);
  static_assert(4 * f32w_wave(2) <= 64 * 1024, "no more LDS than a kernel gets without asking");
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), (size_t)lds, ctx->stream, a.A, a.X, a.M, a.Kdim, a.Ncols, pl.units, pl.rest, pl.whole,
                     pl.stages_per_split, pl.tiles_m, pl.magic_round, pl.magic_tiles_m, a, pl, ctx->splitk_partials, ctx->splitk_counters);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("gemm_f32(waves): launch failed: %s", hipGetErrorString(e)); return false; }
  launched = true;
  return true;
}

}  // namespace dnnrt
