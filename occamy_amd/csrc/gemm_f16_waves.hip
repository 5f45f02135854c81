// fp16 matrix products of at most a tile per compute unit: row-major A[M,K], B stored [K,N] or [N,K], batched, bias / residual /
// GELU behind them (the forms of gemm_f16_dma.hip).
//
// What bounds such a product is a chain of latencies, and in gemm_f16_dma.hip most of it is the loop: a barrier, LDS reads and
// their round trip per 64 k, every operand read by two wavefronts.  Here each of the four wavefronts owns the whole tile, 64 columns
// and 64 or 32 rows, for a quarter of the reduction: a ring of two or three stages of 32 k that nobody else touches, so no
// barrier, every operand read once, 16 MFMAs per stage and wavefront from 12 reads; the four sums meet in LDS at the end, where each lane gets eight
// neighbouring columns of two rows or one, bias and residual having been requested behind the ring's first loads.
//
// Time of a workgroup, 384 x 768 x 2304 (us): set-up 0.5, first data 1.0, six stages 2.5, sums 0.6, epilogue and code fetched on the way 1.0.
// Rings of four stages gained in the loop what they lost waiting for the first data; 96 rows per tile cost 1.2 more per
// launch and never paid.  32 rows are taken where they spare a split reduction its hand-over, or make one of it with half the
// bytes (us, 64 rows alone and with 32): 384 rows, 768 x 768 6.4 -> 5.2; 128 rows, 768 x 2304 6.7 -> 5.3, 768 x 3072 7.1 -> 5.6,
// 3072 x 768 9.3 -> 7.9; 16 rows 6.0 -> 5.0, 6.2 -> 5.5, 8.4 -> 6.8; BERT at 384 tokens 564 -> 548.  K x N, us on gemm_f16_dma.hip
// -> here with 64 rows, back to back on one card: 384 rows, 768 x 2304 7.0 -> 6.6; 3072 x 768 11.2 -> 10.1.
#include "gemm_f16.h"
#include "partials.h"

#include <type_traits>

namespace dnnrt {

typedef _Float16 gw_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 gw_half4 __attribute__((ext_vector_type(4)));
typedef short gw_short4 __attribute__((ext_vector_type(4)));
typedef float gw_floatx16 __attribute__((ext_vector_type(16)));
typedef float gw_floatx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *gw_lds;

[[maybe_unused]] constexpr unsigned GW_OUT_OF_RANGE = 0x80000000u;  // above every num_records used here: reads as zeros
constexpr int GW_BK = 32;                      // k of a stage
constexpr int gw_ring(int tm) { return tm == 2 ? 2 : 3; }                       // stages of a wavefront's ring
constexpr int gw_stage(int tm) { return (64 + 32 * tm) * GW_BK * 2; }            // bytes of a stage
constexpr int gw_wave(int tm) { return tm == 2 ? 64 * 64 * 4 : 3 * gw_stage(1); }  // a wavefront's LDS: its ring and, later, its sums

template <int N>
__device__ __forceinline__ void gw_wait_vmcnt() {  // LDS accesses stay on their side of it
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void gw_wait_lgkm() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
  asm volatile("" ::: "memory");
}

#if __HIP_DEVICE_COMPILE__
// ds_read_b64_tr_b16 at LDS address `at` + OFFSET.  By hand: ahead of the builtin the compiler waits for every load into LDS
// that is still on its way (vmcnt 0), and so for the whole ring.  It knows nothing of this read either: the value is there
// behind the next wait for lgkmcnt, and gw_arrived() ties its uses to that place.  Nothing keeps the compiler from copying or
// spilling the register in between; that it does not, along every branch, is looked up in its output by
// tests/test_untracked_reads.py, which is to be run again with another compiler.
template <int OFFSET>
__device__ __forceinline__ gw_short4 gw_read_tr(unsigned at) {
  gw_short4 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(at), "i"(OFFSET) : "memory");
  return v;
}
#endif
template <class T>
__device__ __forceinline__ void gw_arrived(T &v) {
  asm volatile("" : "+v"(v));
}

// Tiles of 64 columns n and 32 TM rows m; B_KC: B stored [N,K].  The arguments in front of the struct are in registers when a
// wavefront starts: all that the ring's first loads need, so that nothing waits for the rest, which comes 0.45 us later
// (a BERT-base over 384 tokens, 48 of its 88 launches here and in gemm_f16_dma.hip, 541 -> 530 us).
template <bool B_KC, int TM>
__global__ __launch_bounds__(256, 2) void gemm_f16_waves_kernel(const __half *A, const __half *B, int64_t az, int64_t bz, int M, int N, int K, int tiles,
                                                                unsigned magic_tiles_m, int steps_per_split, const GemmF16Args args, int splits) {
#if __HIP_DEVICE_COMPILE__
  GemmF16Args a = args;
  a.M = M; a.N = N; a.K = K; a.steps_per_split = steps_per_split;
  constexpr int NS = gw_ring(TM), FM = 32 * TM, STAGE = gw_stage(TM), WAVE_LDS = gw_wave(TM);
  constexpr int M_L = FM / 16, L = 4 + M_L;  // loads of a stage
  static_assert(NS * STAGE <= WAVE_LDS && FM * 64 * 4 <= WAVE_LDS, "a wavefront's ring and, later, its sums");
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int per_xcd = (tiles + 7) >> 3;  // consecutive tiles (all rows m of one column range) on one XCD share B in its L2
  const int tile = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || tile >= tiles) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int tiles_m = (a.M + FM - 1) / FM, tile_n = div_magic(tile, tiles_m, magic_tiles_m), tile_m = tile - tile_n * tiles_m;
  const int n0 = tile_n * 64, m0 = tile_m * FM, z = blockIdx.z;
  char *ring = smem + wave * WAVE_LDS;

  // ---- this wavefront's stages: every fourth, so that the four read neighbouring rows of B and the same lines of the operands' k-contiguous rows
  // at a time (a quarter each in a run: BERT-base over 384 tokens 526 -> 511 us) ----
  const int stages = (a.K + GW_BK - 1) / GW_BK;
  const int s_beg = (int)blockIdx.y * a.steps_per_split, s_end = min(stages, s_beg + a.steps_per_split);
  const int my_beg = s_beg + wave, nk = max(0, (s_end - my_beg + 3) >> 2);

  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(A) + (int64_t)z * az, 0, 2 * a.M * a.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(B) + (int64_t)z * bz, 0, 2 * a.K * a.N, 0x00020000);

  // ---- loader constants: byte offset of this lane's chunk, and the k of the stage it belongs to ----
  // k-contiguous rows: 64 bytes a row, 16-byte chunk c of row r at c ^ ((r >> 2) & 3); sixteen rows per instruction
  const int ch_k = 8 * ((lane & 3) ^ ((lane >> 4) & 3));
  // [K,N]: 128 bytes a row of k, chunk c of row k at c ^ swz(k); eight rows per instruction
  const int row_k = lane >> 3, swz_k = ((row_k >> 1) & 3) * 2;
  unsigned m_off[M_L], n_off[4];
#pragma unroll
  for (int i = 0; i < M_L; i++) {
    const int r = 16 * i + (lane >> 2);
    m_off[i] = m0 + r < a.M ? 2u * (unsigned)((m0 + r) * a.K + ch_k) : GW_OUT_OF_RANGE;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    [[maybe_unused]] const int r = 16 * i + (lane >> 2);
    if constexpr (B_KC) {
      n_off[i] = n0 + r < a.N ? 2u * (unsigned)((n0 + r) * a.K + ch_k) : GW_OUT_OF_RANGE;
    } else {
      const int n = n0 + 8 * ((lane & 7) ^ swz_k);
      n_off[i] = n < a.N ? 2u * (unsigned)((8 * i + row_k) * a.N + n) : GW_OUT_OF_RANGE;
    }
  }
  int l_k = GW_BK * my_beg, l_slot = 0;
  auto issue_stage = [&]() {
    char *Ns = ring + l_slot * STAGE, *Ms = Ns + 64 * GW_BK * 2;
    const bool tail = l_k + GW_BK > a.K;  // the reduction's last, partial stage
    const bool m_past = tail && l_k + ch_k >= a.K;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const bool past = B_KC ? m_past : tail && l_k + 8 * i + row_k >= a.K;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (gw_lds)(Ns + 1024 * i), 16, past ? GW_OUT_OF_RANGE : n_off[i], B_KC ? 2 * l_k : 2 * l_k * a.N, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < M_L; i++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (gw_lds)(Ms + 1024 * i), 16, m_past ? GW_OUT_OF_RANGE : m_off[i], 2 * l_k, 0, 0);
    l_k += 4 * GW_BK;
    l_slot = l_slot + 1 == NS ? 0 : l_slot + 1;
  };

  // ---- operand fetch --------------------------------------------------------
  const unsigned ld_k[2] = {(unsigned)(l32 * 64 + 16 * (half ^ ((l32 >> 2) & 3))), (unsigned)(l32 * 64 + 16 * ((2 + half) ^ ((l32 >> 2) & 3)))};
  [[maybe_unused]] unsigned tr_off[2][2];  // [K,N]: sub-step 0, k 8 * half + 4 t .. + 3
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int k = 8 * half + 4 * t + ((lane & 15) >> 2), n = 32 * i + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
      tr_off[i][t] = (unsigned)(k * 128 + (((n >> 3) ^ (((k >> 1) & 3) * 2)) * 16) + (n & 7) * 2);
    }
  gw_half8 fm[2][2][TM], fn[2][2][2];  // [set][16 k][block]: two stages' operands
  [[maybe_unused]] gw_short4 tr[2][2][2][2];  // [K,N]: the halves of fn
  int c_slot = 0;
  auto read_stage = [&](auto set_c) {
    constexpr int S = decltype(set_c)::value;
    const char *Ns = ring + c_slot * STAGE, *Ms = Ns + 64 * GW_BK * 2;
    c_slot = c_slot + 1 == NS ? 0 : c_slot + 1;
#pragma unroll
    for (int sub = 0; sub < 2; sub++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        if constexpr (B_KC) {
          fn[S][sub][i] = *reinterpret_cast<const gw_half8 *>(Ns + ld_k[sub] + i * 2048);
        } else {
          const unsigned at = (unsigned)(size_t)(gw_lds)Ns;  // sixteen rows further on the swizzle is the same
          tr[S][sub][i][0] = sub ? gw_read_tr<2048>(at + tr_off[i][0]) : gw_read_tr<0>(at + tr_off[i][0]);
          tr[S][sub][i][1] = sub ? gw_read_tr<2048>(at + tr_off[i][1]) : gw_read_tr<0>(at + tr_off[i][1]);
        }
      }
#pragma unroll
    for (int sub = 0; sub < 2; sub++)
#pragma unroll
      for (int j = 0; j < TM; j++) fm[S][sub][j] = *reinterpret_cast<const gw_half8 *>(Ms + ld_k[sub] + j * 2048);
  };

  gw_floatx16 acc[2][TM];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < TM; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
#pragma unroll
  for (int i = 0; i < NS; i++)
    if (i < nk) issue_stage();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // The other arguments, all at once: read where they are used, each is waited for there.
  asm volatile("" : "+s"(a.bias), "+s"(a.C), "+s"(a.c_sm), "+s"(a.cz), "+s"(a.yz), "+s"(a.Out), "+s"(a.alpha), "+s"(a.beta), "+s"(a.act), "+s"(a.act_coef),
               "+s"(a.partials), "+s"(a.counters), "+s"(splits));
  // What the lane finishes: eight columns out_n .. + 7 of the rows out_m + 32 o.  Bias and residual are requested behind
  // the ring's first loads; the counted waits below are for the loads of the ring alone, these make the first of them stricter.
  const int out_m = m0 + (tid >> 3), out_n = n0 + 8 * (tid & 7);
  const gw_half4 zero4 = {(_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
  gw_half4 bias4[2] = {zero4, zero4}, c4[TM][2];
  if (a.bias) {
#pragma unroll
    for (int q = 0; q < 2; q++) bias4[q] = *reinterpret_cast<const gw_half4 *>(reinterpret_cast<const _Float16 *>(a.bias) + min(out_n + 4 * q, a.N - 4));
  }
  if (a.C) {
    const _Float16 *Cg = reinterpret_cast<const _Float16 *>(a.C) + (int64_t)z * a.cz;
#pragma unroll
    for (int o = 0; o < TM; o++)
#pragma unroll
      for (int q = 0; q < 2; q++) c4[o][q] = *reinterpret_cast<const gw_half4 *>(Cg + (int64_t)min(out_m + 32 * o, a.M - 1) * a.c_sm + min(out_n + 4 * q, a.N - 4));
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  // ---- the reduction: nobody shares a ring, so there is no barrier ------------
  auto multiply = [&](auto set_c, auto sub_c) {
    constexpr int S = decltype(set_c)::value, sub = decltype(sub_c)::value;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < TM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fn[S][sub][i], fm[S][sub][j], acc[i][j], 0, 0, 0);
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  auto landed = [&](int behind) {  // the oldest stage in flight has landed, up to NS - 1 behind it may still be on their way
    if (behind >= NS - 1) gw_wait_vmcnt<(NS - 1) * L>();
    else if (NS > 2 && behind == 1) gw_wait_vmcnt<L>();
    else gw_wait_vmcnt<0>();
  };
  // One stage, its operands in set S or on their way there; `ahead` follow it.
  auto step = [&](auto set_c, int ahead) {
    constexpr int S = decltype(set_c)::value;
    gw_wait_lgkm();  // its operands are here: its slot is free
    if constexpr (!B_KC) {
#pragma unroll
      for (int sub = 0; sub < 2; sub++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
          gw_arrived(tr[S][sub][i][0]);
          gw_arrived(tr[S][sub][i][1]);
          fn[S][sub][i] = __builtin_bit_cast(gw_half8, __builtin_shufflevector(tr[S][sub][i][0], tr[S][sub][i][1], 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
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
  if constexpr (!B_KC) {
    gw_wait_lgkm();  // no read is on its way, whatever the branches above: the registers are free
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- the four wavefronts' sums meet in LDS: [m][n] in fp32, 16-byte chunk c of row m at c ^ (m & 15) ----
  // register r of block (i, j): n = 32 i + 8 (r / 4) + 4 half + r % 4, m = 32 j + l32
#pragma unroll
  for (int j = 0; j < TM; j++)
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const gw_floatx4 v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        *reinterpret_cast<gw_floatx4 *>(ring + (32 * j + l32) * 256 + 16 * ((8 * i + 2 * g + half) ^ (l32 & 15))) = v;
      }
  __syncthreads();
  constexpr int E = 8 * TM;
  float v[E];
#pragma unroll
  for (int o = 0; o < TM; o++)
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int m = (tid >> 3) + 32 * o;
      const char *at = smem + m * 256 + 16 * ((2 * (tid & 7) + q) ^ (m & 15));
      gw_floatx4 s = *reinterpret_cast<const gw_floatx4 *>(at);
#pragma unroll
      for (int w = 1; w < 4; w++) s += *reinterpret_cast<const gw_floatx4 *>(at + w * WAVE_LDS);
#pragma unroll
      for (int e = 0; e < 4; e++) v[8 * o + 4 * q + e] = s[e];
    }

  // ---- a split reduction: the hand-over of the fp32 kernels (igemm_f32_small.hip states what it rests on) ----
  if (splits > 1) {
    const unsigned t = (unsigned)z * (unsigned)tiles + (unsigned)tile;
    const __amdgpu_buffer_rsrc_t parts = part_rsrc(a.partials);
    const unsigned mine = 16u * (unsigned)tid, first_part = t * (unsigned)splits * (FM * 256u);
#pragma unroll
    for (int e = 0; e < E; e += 4) part_store(parts, mine + 1024 * e, first_part + blockIdx.y * (FM * 256u), part_floatx4{v[e], v[e + 1], v[e + 2], v[e + 3]});
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    volatile unsigned *arrived = reinterpret_cast<unsigned *>(smem);
    if (tid == 0) *arrived = __hip_atomic_fetch_add(&a.counters[t], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived != (unsigned)splits - 1) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (tid == 0) __hip_atomic_store(&a.counters[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int e = 0; e < E; e++) v[e] = 0.f;
    for (int y0 = 0; y0 < splits; y0 += 4) {  // four parts requested at a time, added in split order
      part_floatx4 p[4][E / 4];
#pragma unroll
      for (int y = 0; y < 4; y++)
#pragma unroll
        for (int e = 0; e < E; e += 4)
          p[y][e / 4] = part_load<part_floatx4>(parts, y0 + y < splits ? mine + 1024 * e : PART_NONE, first_part + (unsigned)min(y0 + y, splits - 1) * (FM * 256u));
#pragma unroll
      for (int y = 0; y < 4; y++)
#pragma unroll
        for (int e = 0; e < E; e++) v[e] += p[y][e / 4][e % 4];
    }
  }

  // ---- epilogue: act((alpha acc + bias) + beta C) in fp32, one rounding -------
  auto finish = [&](auto mode_c) {
    constexpr int ACT = decltype(mode_c)::value;
#pragma unroll
    for (int o = 0; o < TM; o++) {
      const int m = out_m + 32 * o;
      gw_half8 w;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        float x = a.alpha * v[8 * o + e] + (float)bias4[e / 4][e % 4];
        if (a.C) x += a.beta * (float)c4[o][e / 4][e % 4];
        w[e] = (_Float16)apply_act(x, ACT, a.act_coef);
      }
      if (m < a.M && out_n < a.N) *reinterpret_cast<gw_half8 *>(reinterpret_cast<_Float16 *>(a.Out) + (int64_t)z * a.yz + (int64_t)m * a.N + out_n) = w;
    }
  };
  if (a.act == ACT_GELU) finish(std::integral_constant<int, ACT_GELU>{});
  else finish(std::integral_constant<int, DNNRT_ACT_IDENTITY>{});
#endif
}

template <bool B_KC, int TM>
static bool launch_one(const dnnrtContext *ctx, const GemmF16Args &g, const dim3 &grid, int tiles) {
  constexpr int SMEM = 4 * gw_wave(TM);
  if constexpr (SMEM > 64 * 1024) {
    static LdsRaised raised;
    if (!raise_lds(raised, ctx->device, reinterpret_cast<const void *>(&gemm_f16_waves_kernel<B_KC, TM>), SMEM)) {
      set_error("matmul(fp16): cannot reserve %d bytes of LDS", SMEM);
      return false;
    }
  }
  hipLaunchKernelGGL((gemm_f16_waves_kernel<B_KC, TM>), grid, dim3(256), SMEM, ctx->stream, g.A, g.B, g.az, g.bz, g.M, g.N, g.K, tiles,
                     magic_of((int)ceil_div(g.M, 32 * TM)), g.steps_per_split, g, (int)grid.y);
  return true;
}

bool launch_gemm_f16_waves(const dnnrtContext *ctx, const GemmF16Args &args, int Z, int rows, int splits) {
  GemmF16Args g = args;
  const int tiles = (int)(ceil_div(g.M, rows) * ceil_div(g.N, 64)), stages = (int)ceil_div(g.K, GW_BK);
  g.steps_per_split = (int)ceil_div(stages, splits);
  splits = (int)ceil_div(stages, g.steps_per_split);  // no empty split: every arrival carries a partial tile
  if (splits > 1 && ((int64_t)tiles * Z * splits * rows * 256 > ctx->splitk_partial_bytes || (int64_t)tiles * Z > ctx->splitk_max_tiles)) {
    set_error("matmul(fp16): %d parts of %d tiles do not fit the reduction scratch", splits, tiles);
    return false;
  }
  const dim3 grid((unsigned)(ceil_div(tiles, 8) * 8), (unsigned)splits, (unsigned)Z);
  const bool done = g.b_sk == 1 ? (rows == 64 ? launch_one<true, 2>(ctx, g, grid, tiles) : launch_one<true, 1>(ctx, g, grid, tiles))
                                : (rows == 64 ? launch_one<false, 2>(ctx, g, grid, tiles) : launch_one<false, 1>(ctx, g, grid, tiles));
  if (!done) return false;
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("matmul(fp16): launch failed: %s", hipGetErrorString(e)); return false; }
  return true;
}

}  // namespace dnnrt
