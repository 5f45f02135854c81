// fp16 matrix products whose operands go from global memory straight into LDS (buffer_load_dwordx4 ... lds), for row-major
// A[M,K] and B stored [K,N] (a Linear layer's weights as they come) or [N,K], batched, bias / residual / GELU behind them.
//
// D[n, m] = sum_k B[k, n] A[m, k] on v_mfma_f32_32x32x16_f16: rows of a block are output columns n, so that a lane holds
// four consecutive n of one m.  A step is 64 k.  A's rows lie in LDS as in conv_f16_dma.hip (128-byte rows, 16-byte chunk c
// of row r at c ^ ((r >> 1) & 7)), and so do B's when it is stored [N,K].  Stored [K,N] its rows lie in LDS as in memory,
// [64 k][n], and an operand (eight consecutive k of one n) comes out of two transposing reads, ds_read_b64_tr_b16: lane
// i of sixteen asks for four n of row k + i / 4 and receives element i of four consecutive rows.  The chunks of a row are
// swizzled so that the four rows of such a read lie in different banks.
//
// What bounds it: at a transformer's sizes (16 to a few hundred rows, 0.1 .. 2 GFLOP) a chain of latencies per step, its
// barrier, LDS reads and requests; the matrix pipes are busy for a tenth of the time.  Hence 64x64 tiles, all of a step's
// operands read one step ahead (0.56 -> 0.37 us per step against reads a 16-k sub-step ahead; 0.30 since the transposing reads
// no longer wait for the whole ring, gd_read_tr), and reductions split over workgroups where tiles are few (partial tiles through the handle's scratch,
// the last to arrive adds them in split order; nobody waits).  128x128 tiles on eight wavefronts take the products of
// thousands of rows (4096 cubed: 650 TFLOP/s, 333 us on 64x64 tiles, 212 on these).
// Against gemm_f16.hip's kernel, which keeps what is not aligned (K x N -> us before, now): 384 rows, 768 x 2304 19.4 -> 7.0,
// 768 x 768 15.9 -> 7.0, 768 x 3072 + GELU 24.7 -> 9.1, 3072 x 768 26.7 -> 11.2; 2048 rows, 768 x 2304 18.2.  Products of at most a tile per
// compute unit go to gemm_f16_waves.hip.
#include "gemm_f16.h"
#include "partials.h"

#include <algorithm>
#include <type_traits>

namespace dnnrt {

typedef _Float16 gd_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 gd_half4 __attribute__((ext_vector_type(4)));
typedef short gd_short4 __attribute__((ext_vector_type(4)));
typedef short gd_short8 __attribute__((ext_vector_type(8)));
typedef float gd_floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void *gd_lds;

[[maybe_unused]] constexpr unsigned GD_OUT_OF_RANGE = 0x80000000u;  // above every num_records used here: reads as zeros

template <int N, int LGKM = 15>
__device__ __forceinline__ void gd_wait() {  // s_waitcnt vmcnt(N) lgkmcnt(LGKM), 15: any
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (LGKM << 8));
}
__device__ __forceinline__ void gd_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

#if __HIP_DEVICE_COMPILE__
// ds_read_b64_tr_b16 at LDS address `at` + OFFSET.  By hand: ahead of the builtin the compiler waits for every load into LDS
// that is still on its way (vmcnt 0), and so for the whole ring.  It knows nothing of this read either: the value is there
// behind the next wait for lgkmcnt, and gd_arrived() ties its uses to that place.  Nothing keeps the compiler from copying or
// spilling the register in between; that it does not, along every branch, is looked up in its output by
// tests/test_untracked_reads.py, which is to be run again with another compiler.
template <int OFFSET>
__device__ __forceinline__ gd_short4 gd_read_tr(unsigned at) {
  gd_short4 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(at), "i"(OFFSET) : "memory");
  return v;
}
#endif
template <class T>
__device__ __forceinline__ void gd_arrived(T &v) {
  asm volatile("" : "+v"(v));
}

// FN x FM: columns n and rows m of a workgroup's tile, over WN x WM wavefronts; NS ring stages; B_KC: B stored [N,K].  What the
// ring's first loads need stands in front of the struct and is in registers when a wavefront starts; the rest comes 0.45 us later.
template <int FN, int FM, int WN, int WM, int NS, bool B_KC>
__global__ __launch_bounds__(64 * WN * WM) void gemm_f16_dma_kernel(const __half *A, const __half *B, int64_t az, int64_t bz, int M, int N, int K, int tiles,
                                                                     unsigned magic_tiles_m, int steps_per_split, const GemmF16Args args, int splits) {
#if __HIP_DEVICE_COMPILE__
  GemmF16Args a = args;
  a.M = M; a.N = N; a.K = K; a.steps_per_split = steps_per_split;
  constexpr int NW = WN * WM, NT = 64 * NW, TN = FN / WN / 32, TM = FM / WM / 32;
  constexpr int STAGE = (FN + FM) * 128;
  constexpr int N_L = FN / 8 / NW, M_L = FM / 8 / NW, L = N_L + M_L;  // loads per wavefront and step
  constexpr int NCH = FN / 8, NROWS = 64 / NCH;                       // [K,N]: chunks per row, rows per load
  static_assert(FN % (8 * NW) == 0 && FM % (8 * NW) == 0 && TN >= 1 && TM >= 1, "tile does not divide over the wavefronts");
  static_assert(FN == 64 || FN == 128, "the swizzles below");
  constexpr int CROW = FN + 8;  // halfs per row of the output staging tile
  static_assert(FM * CROW * 2 <= NS * STAGE, "the output tile is staged in the operand ring");
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int per_xcd = (tiles + 7) >> 3;  // consecutive tiles (all rows m of one column range) on one XCD share B in its L2
  const int tile = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || tile >= tiles) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int wn0 = (wave / WM) * (FN / WN), wm0 = (wave % WM) * (FM / WM);
  const int tiles_m = (a.M + FM - 1) / FM, tile_n = div_magic(tile, tiles_m, magic_tiles_m), tile_m = tile - tile_n * tiles_m;
  const int n0 = tile_n * FN, m0 = tile_m * FM, z = blockIdx.z;

  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(A) + (int64_t)z * az, 0, 2 * a.M * a.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half *>(B) + (int64_t)z * bz, 0, 2 * a.K * a.N, 0x00020000);

  // ---- loader constants: byte offset of this lane's chunk, and the k of the step it belongs to ----
  unsigned m_off[M_L], n_off[N_L];
  const int ch_k = (lane & 7) ^ (((8 * wave + (lane >> 3)) >> 1) & 7);  // k-contiguous rows: the same for every load of the wavefront
#pragma unroll
  for (int i = 0; i < M_L; i++) {
    const int m = m0 + 8 * (wave + i * NW) + (lane >> 3);
    m_off[i] = m < a.M ? 2u * (unsigned)(m * a.K + ch_k * 8) : GD_OUT_OF_RANGE;
  }
  auto swz = [](int k) { return FN == 64 ? ((k >> 1) & 3) * 2 : (k & 3) * 2; };  // [K,N]: chunk c of row k at c ^ swz(k)
#pragma unroll
  for (int i = 0; i < N_L; i++) {
    if constexpr (B_KC) {
      const int n = n0 + 8 * (wave + i * NW) + (lane >> 3);
      n_off[i] = n < a.N ? 2u * (unsigned)(n * a.K + ch_k * 8) : GD_OUT_OF_RANGE;
    } else {
      const int k = NROWS * (wave + i * NW) + lane / NCH, n = n0 + 8 * ((lane % NCH) ^ swz(k));
      n_off[i] = n < a.N ? 2u * (unsigned)(k * a.N + n) : GD_OUT_OF_RANGE;
    }
  }
  const int steps = (a.K + 63) >> 6;
  const int s_beg = (int)blockIdx.y * a.steps_per_split, s_end = min(steps, s_beg + a.steps_per_split);
  int l_k = 64 * s_beg, l_stage = 0;
  auto issue_loads = [&]() {  // the next step, into the next stage
    char *Ns = smem + l_stage * STAGE, *Ms = Ns + FN * 128;
    const bool tail = l_k + 64 > a.K;  // the reduction's last, partial step
#pragma unroll
    for (int i = 0; i < N_L; i++) {
      unsigned off = n_off[i];
      if (tail && l_k + (B_KC ? ch_k * 8 : NROWS * (wave + i * NW) + lane / NCH) >= a.K) off = GD_OUT_OF_RANGE;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (gd_lds)(Ns + 1024 * (wave + i * NW)), 16, off, B_KC ? 2 * l_k : 2 * l_k * a.N, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < M_L; i++) {
      unsigned off = m_off[i];
      if (tail && l_k + ch_k * 8 >= a.K) off = GD_OUT_OF_RANGE;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (gd_lds)(Ms + 1024 * (wave + i * NW)), 16, off, 2 * l_k, 0, 0);
    }
    l_k += 64;
    l_stage = l_stage + 1 == NS ? 0 : l_stage + 1;
  };

  gd_floatx16 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; i++)
#pragma unroll
    for (int j = 0; j < TM; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  // ---- operand fetch --------------------------------------------------------
  const unsigned ld_m0 = (unsigned)((FN + wm0 + l32) * 128 + ((half ^ ((l32 >> 1) & 7)) * 16));
  [[maybe_unused]] const unsigned ld_n0 = (unsigned)((wn0 + l32) * 128 + ((half ^ ((l32 >> 1) & 7)) * 16));
  [[maybe_unused]] unsigned tr_off[TN][2];  // [K,N]: sub-step 0, k 8 * half + 4 t .. + 3
#pragma unroll
  for (int i = 0; i < TN; i++)
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int k = 8 * half + 4 * t + ((lane & 15) >> 2), n = wn0 + 32 * i + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
      tr_off[i][t] = (unsigned)(k * 2 * FN + (((n >> 3) ^ swz(k)) * 16) + (n & 7) * 2);
    }
  gd_half8 fn[2][4][TN], fm[2][4][TM];  // two steps' operands
  [[maybe_unused]] gd_short4 tr[2][4][TN][2];  // [K,N]: the halves of fn
  auto read_step = [&](const char *stage, auto set_c) {
    constexpr int S = decltype(set_c)::value;
#pragma unroll
    for (int sub = 0; sub < 4; sub++) {
#pragma unroll
      for (int i = 0; i < TN; i++) {
        if constexpr (B_KC) {
          fn[S][sub][i] = *reinterpret_cast<const gd_half8 *>(stage + ((ld_n0 ^ (32u * sub)) + i * 4096));
        } else {
          const unsigned at = (unsigned)(size_t)(gd_lds)const_cast<char *>(stage);  // sixteen rows further on the swizzle is the same
#pragma unroll
          for (int t = 0; t < 2; t++) {
            const unsigned from = at + tr_off[i][t];
            tr[S][sub][i][t] = sub == 0 ? gd_read_tr<0>(from) : sub == 1 ? gd_read_tr<32 * FN>(from) : sub == 2 ? gd_read_tr<64 * FN>(from) : gd_read_tr<96 * FN>(from);
          }
        }
      }
#pragma unroll
      for (int j = 0; j < TM; j++) fm[S][sub][j] = *reinterpret_cast<const gd_half8 *>(stage + ((ld_m0 ^ (32u * sub)) + j * 4096));
    }
  };

  // ---- the ring: all NS stages in flight.  A step's operands are read a step ahead, all of them behind the one barrier,
  // so that the LDS round trip runs under the multiplication of the step before and the loads of the step NS ahead.  A
  // wavefront's reads of a stage are done (lgkmcnt 0) before the next barrier, behind which that stage is loaded again.
  static_assert(NS >= 2 && NS <= 4 && (NS - 2) * L < 64, "ring depth");
  constexpr std::integral_constant<int, 0> set0{};
  constexpr std::integral_constant<int, 1> set1{};
  int c_stage = 0;
  auto step_body = [&](auto set_c, auto full_c, int ahead) {  // `ahead` steps follow this one; FULL: NS or more
    constexpr int S = decltype(set_c)::value;
    constexpr bool FULL = decltype(full_c)::value;
    // the next step has landed, NS - 2 behind it may still be on their way; this one's operands are here
    if (FULL) {
      gd_wait<(NS - 2) * L, 0>();
    } else {
      gd_wait<63, 0>();  // whatever the branches below
      if (NS > 3 && ahead > 2) gd_wait<(NS > 3 ? 2 : 0) * L>();
      else if (NS > 2 && ahead > 1) gd_wait<(NS > 2 ? 1 : 0) * L>();
      else gd_wait<0>();
    }
    if constexpr (!B_KC) {
#pragma unroll
      for (int sub = 0; sub < 4; sub++)
#pragma unroll
        for (int i = 0; i < TN; i++) {
          gd_arrived(tr[S][sub][i][0]);
          gd_arrived(tr[S][sub][i][1]);
          fn[S][sub][i] = __builtin_bit_cast(gd_half8, __builtin_shufflevector(tr[S][sub][i][0], tr[S][sub][i][1], 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
    if (FULL || ahead > 0) {
      gd_barrier();
      c_stage = c_stage + 1 == NS ? 0 : c_stage + 1;
      read_step(smem + c_stage * STAGE, std::integral_constant<int, 1 - S>{});
      if (FULL || ahead >= NS) issue_loads();
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int sub = 0; sub < 4; sub++)
#pragma unroll
      for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fn[S][sub][i], fm[S][sub][j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  const int nk = s_end - s_beg, pre = nk < NS ? nk : NS;
#pragma unroll
  for (int q = 0; q < NS; q++)
    if (q < pre) issue_loads();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // The other arguments, all at once: read where they are used, each is waited for there.
  asm volatile("" : "+s"(a.bias), "+s"(a.C), "+s"(a.c_sm), "+s"(a.cz), "+s"(a.yz), "+s"(a.Out), "+s"(a.alpha), "+s"(a.beta), "+s"(a.act), "+s"(a.act_coef),
               "+s"(a.partials), "+s"(a.counters), "+s"(splits));
  // Bias of this lane's columns, behind the ring's first loads: the counted waits are for the loads of the ring alone, these make the
  // first of them stricter.
  gd_half4 bias4[TN][4];
#pragma unroll
  for (int i = 0; i < TN; i++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int n = n0 + wn0 + i * 32 + 8 * g + 4 * half;
      const gd_half4 zero = {(_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
      bias4[i][g] = a.bias ? *reinterpret_cast<const gd_half4 *>(reinterpret_cast<const _Float16 *>(a.bias) + (n < a.N ? n : 0)) : zero;
    }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  {
    if (pre == 1) gd_wait<0>();
    else if (pre == 2) gd_wait<L>();
    else if (pre == 3) gd_wait<(NS > 2 ? 2 : 0) * L>();
    else gd_wait<(NS > 3 ? 3 : 0) * L>();
    gd_barrier();
    read_step(smem, set0);
  }
  {
    int ahead = nk - 1;
    for (; ahead > NS; ahead -= 2) {
      step_body(set0, std::true_type{}, ahead);
      step_body(set1, std::true_type{}, ahead - 1);
    }
#pragma unroll 1
    for (; ahead > 0; ahead -= 2) {
      step_body(set0, std::false_type{}, ahead);
      step_body(set1, std::false_type{}, ahead - 1);
    }
    if (ahead == 0) step_body(set0, std::false_type{}, 0);
  }
  if constexpr (!B_KC) {
    gd_wait<63, 0>();  // no read is on its way, whatever the branches above: the registers are free
    __builtin_amdgcn_sched_barrier(0);
  }
  gd_barrier();  // nobody reads the operand stages any more

  // ---- a split reduction: the hand-over of the fp32 kernels (igemm_f32_small.hip states what it rests on) ----
  if (splits > 1) {
    constexpr int TILE = FN * FM;
    volatile unsigned *arrived = reinterpret_cast<unsigned *>(smem);
    const unsigned t = (unsigned)z * (unsigned)tiles + (unsigned)tile;
    const __amdgpu_buffer_rsrc_t parts = part_rsrc(a.partials);
    const unsigned mine = 16u * (unsigned)tid, first_part = t * (unsigned)splits * (4u * TILE);  // [four registers][thread]
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
      for (int j = 0; j < TM; j++)
#pragma unroll
        for (int g = 0; g < 4; g++)
          part_store(parts, mine + 16 * NT * ((i * TM + j) * 4 + g), first_part + blockIdx.y * (4u * TILE),
                     part_floatx4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]});
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (tid == 0) *arrived = __hip_atomic_fetch_add(&a.counters[t], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived != (unsigned)splits - 1) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
      for (int j = 0; j < TM; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    for (int y0 = 0; y0 < splits; y0 += 4) {  // four parts requested at a time, added in split order
#pragma unroll
      for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++) {
          part_floatx4 p[4][4];
#pragma unroll
          for (int y = 0; y < 4; y++)
#pragma unroll
            for (int g = 0; g < 4; g++)
              p[y][g] = part_load<part_floatx4>(parts, y0 + y < splits ? mine + 16 * NT * ((i * TM + j) * 4 + g) : PART_NONE, first_part + (unsigned)min(y0 + y, splits - 1) * (4u * TILE));
#pragma unroll
          for (int y = 0; y < 4; y++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] += p[y][r >> 2][r & 3];
        }
    }
    if (tid == 0) __hip_atomic_store(&a.counters[t], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();  // everyone has read `arrived`: the output tile goes over it
  }

  // ---- epilogue: act((alpha acc + bias) + beta C) in fp32, one rounding, transposed through LDS to whole rows ----
  // register r of block (i, j): n = n0 + wn0 + 32 i + 8 (r / 4) + 4 half + r % 4, m = m0 + wm0 + 32 j + l32
  _Float16 *Cs = reinterpret_cast<_Float16 *>(smem);  // [FM][CROW]
  const _Float16 *__restrict__ Cg = a.C ? reinterpret_cast<const _Float16 *>(a.C) + (int64_t)z * a.cz : nullptr;
  auto stage_out = [&](auto mode_c) {
    constexpr int ACT = decltype(mode_c)::value;
#pragma unroll
    for (int j = 0; j < TM; j++) {
      const int m = min(m0 + wm0 + 32 * j + l32, a.M - 1);
      gd_half4 c4[TN][4];
      if (Cg) {
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const int n = n0 + wn0 + 32 * i + 8 * g + 4 * half;
            c4[i][g] = *reinterpret_cast<const gd_half4 *>(Cg + (int64_t)m * a.c_sm + (n < a.N ? n : 0));
          }
      }
#pragma unroll
      for (int i = 0; i < TN; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          gd_half4 o;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            float v = a.alpha * acc[i][j][4 * g + e] + (float)bias4[i][g][e];
            if (Cg) v += a.beta * (float)c4[i][g][e];
            o[e] = (_Float16)apply_act(v, ACT, a.act_coef);
          }
          *reinterpret_cast<gd_half4 *>(Cs + (wm0 + 32 * j + l32) * CROW + wn0 + 32 * i + 8 * g + 4 * half) = o;
        }
    }
  };
  if (a.act == ACT_GELU) stage_out(std::integral_constant<int, ACT_GELU>{});
  else stage_out(std::integral_constant<int, DNNRT_ACT_IDENTITY>{});
  __syncthreads();
  _Float16 *__restrict__ Og = reinterpret_cast<_Float16 *>(a.Out) + (int64_t)z * a.yz;
  constexpr int CH = FN / 8;
  static_assert(FM * CH % NT == 0, "output chunks divide over the threads");
#pragma unroll
  for (int o = 0; o < FM * CH / NT; o++) {
    const int id = tid + o * NT, row = id / CH, ch = id - row * CH, m = m0 + row, n = n0 + 8 * ch;
    if (m < a.M && n < a.N) *reinterpret_cast<gd_half8 *>(Og + (int64_t)m * a.N + n) = *reinterpret_cast<const gd_half8 *>(Cs + row * CROW + 8 * ch);
  }
#endif
}

template <int FN, int FM, int WN, int WM, int NS>
static bool launch_gd(const dnnrtContext *ctx, const GemmF16Args &g, int Z, int splits) {
  constexpr int SMEM = NS * (FN + FM) * 128;
  const int64_t tiles = ceil_div(g.M, FM) * ceil_div(g.N, FN);
  const bool kc = g.b_sk == 1;
  if (SMEM > 64 * 1024) {
    static LdsRaised raised[2];
    const void *kernel = kc ? reinterpret_cast<const void *>(&gemm_f16_dma_kernel<FN, FM, WN, WM, NS, true>)
                            : reinterpret_cast<const void *>(&gemm_f16_dma_kernel<FN, FM, WN, WM, NS, false>);
    if (!raise_lds(raised[kc], ctx->device, kernel, SMEM)) {
      set_error("matmul(fp16): cannot reserve %d bytes of LDS", SMEM);
      return false;
    }
  }
  const dim3 grid((unsigned)(ceil_div(tiles, 8) * 8), (unsigned)splits, (unsigned)Z), block(64 * WN * WM);
  const unsigned magic = magic_of((int)ceil_div(g.M, FM));
  if (kc) hipLaunchKernelGGL((gemm_f16_dma_kernel<FN, FM, WN, WM, NS, true>), grid, block, SMEM, ctx->stream, g.A, g.B, g.az, g.bz, g.M, g.N, g.K, (int)tiles, magic,
                             g.steps_per_split, g, (int)grid.y);
  else hipLaunchKernelGGL((gemm_f16_dma_kernel<FN, FM, WN, WM, NS, false>), grid, block, SMEM, ctx->stream, g.A, g.B, g.az, g.bz, g.M, g.N, g.K, (int)tiles, magic,
                             g.steps_per_split, g, (int)grid.y);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("matmul(fp16): launch failed: %s", hipGetErrorString(e)); return false; }
  return true;
}

bool launch_gemm_f16_dma(const dnnrtContext *ctx, const GemmF16Args &args, int Z, bool &launched) {
  launched = false;
  GemmF16Args g = args;
  // row-major A; 16-byte runs along K (A, B stored [N,K]) and N (B stored [K,N], the result, the residual)
  if (g.a_sk != 1 || !g.a_vec || !g.b_vec || g.K % 8 || g.N % 8 || (g.b_sk != 1 && g.b_sn != 1) || (g.act != ACT_GELU && g.act != DNNRT_ACT_IDENTITY) ||
      (int64_t)g.M * g.K >= (1ll << 30) || (int64_t)g.K * g.N >= (1ll << 30) || !aligned16(g.Out) || g.yz % 8 || (reinterpret_cast<uintptr_t>(g.bias) & 7u) ||
      (g.C && ((reinterpret_cast<uintptr_t>(g.C) & 7u) || g.c_sm % 4 || g.cz % 4)))
    return true;
  // Estimated microseconds, fitted on 16 .. 4096 rows and 768 / 3072 columns and channels: a step of 64 k takes a compute
  // unit t1 with one workgroup, tm per workgroup with several; a split's hand-over takes 3 and more with its parts.
  static const struct { int fn, fm; double t1, tm; } shapes[] = {{64, 64, 0.30, 0.23}, {128, 128, 0.56, 0.80}};
  const int steps = (int)ceil_div(g.K, 64);
  int best = -1, best_splits = 1;
  double best_cost = 0;
  for (int i = 0; i < 2; i++) {
    const int64_t tiles = ceil_div(g.M, shapes[i].fm) * ceil_div(g.N, shapes[i].fn) * Z;
    if (tiles > (1 << 28)) continue;
    for (int s = 1; s <= 16 && s <= steps; s++) {
      if (s > 1 && (ctx->splitk_shared || tiles > ctx->splitk_max_tiles || tiles * s * shapes[i].fn * shapes[i].fm * 4 > ctx->splitk_partial_bytes)) break;
      const int per = (int)ceil_div(steps, s);
      if (ceil_div(steps, per) != s) continue;  // no empty split: every arrival carries a partial tile
      const int64_t n = ceil_div(tiles * s, ctx->num_cu);
      const double cost = per * (n > 1 ? fmax((double)n * shapes[i].tm, shapes[i].t1) : shapes[i].t1) + (s > 1 ? 2.9 + 0.32 * s : 0);
      if (best < 0 || cost < best_cost) { best = i; best_cost = cost; best_splits = s; g.steps_per_split = per; }
    }
  }
  // The kernel whose wavefronts share the reduction: a stage of 32 k takes each of the four 0.43, with tiles of 32 rows 0.36, what
  // comes before and after them 0.3 more than here, a split's hand-over 2.3 and 0.25 per part (0.13).  One workgroup per compute
  // unit of the XCD that gets the most tiles: with two it is alone as fast (384 x 768 x 3072 8.3 us either way) and
  // slower in a network (BERT-base over 384 tokens 513 against 510).
  const int stages = (int)ceil_div(g.K, 32);
  int waves_splits = 0, waves_rows = 0;
  for (int rows = 64; rows >= 32; rows -= 32) {
    const int64_t tiles = ceil_div(g.M, rows) * ceil_div(g.N, 64) * Z;
    for (int s = 1; s <= 16 && s <= stages && ceil_div(tiles, 8) * s <= std::max(ctx->num_cu / 8, 1); s++) {
      if (s > 1 && (ctx->splitk_shared || tiles > ctx->splitk_max_tiles || tiles * s * rows * 256 > ctx->splitk_partial_bytes)) break;
      const int per = (int)ceil_div(stages, s);
      if (ceil_div(stages, per) != s) continue;
      const double cost = 0.3 + (rows == 64 ? 0.43 : 0.36) * (double)ceil_div(per, 4) + (s > 1 ? 2.3 + rows / 256.0 * s : 0);
      if (best < 0 || cost < best_cost) { best = 2; best_cost = cost; waves_splits = s; waves_rows = rows; }
    }
  }
  if (best < 0) return true;
  launched = true;
  if (waves_splits) return launch_gemm_f16_waves(ctx, g, Z, waves_rows, waves_splits);
  switch (best) {
    case 0: return launch_gd<64, 64, 2, 2, 4>(ctx, g, Z, best_splits);
    default: return launch_gd<128, 128, 2, 4, 4>(ctx, g, Z, best_splits);
  }
}

}  // namespace dnnrt
