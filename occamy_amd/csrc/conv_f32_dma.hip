// fp32 convolution (any filter, stride and padding, filters C,R,S,K) as an implicit GEMM on v_mfma_f32_32x32x2f32 whose
// operands go from global memory straight into LDS (buffer_load_dword / dwordx4 ... lds).
//
// D[k_out, pixel] = sum_k A[k, k_out] * X[k, pixel].  Both operands are kept in LDS as [k][k_out] and [k][pixel], the
// way they lie in memory, in a ring of stages of 16 or 32 k.  One load instruction fills 64 (dword) or 256 (dwordx4)
// consecutive words of a stage; where each lane's word comes from is its buffer offset alone, so im2col costs a few
// integer instructions per step and wavefront and no vector register, LDS store or mask: padding, pixels past the end
// and filters past K_out are lanes whose offset has bit 31 set, which read zeros.  A 32x32x2 fp32 MFMA occupies a
// SIMD's matrix pipe for 64 cycles (157 TFLOP/s over the chip), so one wavefront per SIMD has 16 issue slots per MFMA
// for all of that, and a second workgroup on the compute unit covers the barriers.
//
// A wavefront's blocks interleave: row i of block t is k_out TM * i + t, column j of block u is pixel TN * j + u.  One
// 8-byte LDS read then feeds two blocks, and a lane's two columns are neighbouring pixels: results leave (and the
// residual comes) as 8-byte accesses, 256 contiguous bytes per half wavefront.
//
// What bounds it: the matrix pipes, and how evenly the tiles fill 256 compute units.  The launcher picks the tile from
// a cost estimate, and the tiles left over after the last full round are each split along the reduction over several
// workgroups (partial tiles through the handle's scratch, the last to arrive adds them in split order; nobody waits).
//
// Measured against the register-staged kernels of igemm_f32.hip / igemm_f32_3x3.hip, which keep the other filter layout,
// groups and transposed products (microseconds; TFLOP/s of 157): 64 -> 64 3x3 at 56x56, 32 images 190 -> 66 (112);
// 256 -> 64 1x1 there 110 -> 34; 256 -> 256 3x3 at 38x38, 3 images 111 -> 51 (100); 256 -> 512 3x3 at 56x56, 2 images
// 201 -> 117 (126); 1024 -> 1024 3x3 at 7x7, 2 images 42 -> 32.  ResNet-50 at 32 images 4.92 -> 2.7 ms.
#include "igemm_f32.h"
#include "partials.h"

#include <type_traits>

namespace dnnrt {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));  // two words at any word address
typedef __attribute__((address_space(3))) void *lds_ptr;

[[maybe_unused]] constexpr unsigned D32_OUT_OF_RANGE = 0x80000000u;  // above every num_records used here: reads as zeros
constexpr int D32_BK = 16;

// How a launch is cut: workgroups 0 .. units - 1 (a multiple of 8) are the split tiles' parts, the rest whole tiles.
struct Dma32Plan {
  int tiles_m, whole, rest, splits, round, units, steps, steps_per_split;  // round: workgroups per part number
  bool neighbours;  // how the parts go to the XCDs (xcd_tile())
  unsigned magic_tiles_m, magic_round;
};

// s_waitcnt vmcnt(N), lgkmcnt as given (15: any); gfx9 encoding.
template <int N, int LGKM = 15>
__device__ __forceinline__ void d32_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (LGKM << 8));
}
#if __HIP_DEVICE_COMPILE__
template <int BYTES>
__device__ __forceinline__ void d32_load(__amdgpu_buffer_rsrc_t rsrc, lds_ptr to, unsigned voff, int soff) {
  if constexpr (BYTES == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, to, 16, voff, soff, 0, 0);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, to, 4, voff, soff, 0, 0);
}
#endif
// A barrier the compiler neither adds waits to nor moves LDS accesses across.
__device__ __forceinline__ void d32_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// TAPS: the filter has more than one tap, or padding.  Reduction order: with C4 (C a multiple of 4) tap by tap, the
// channels of a tap in a row, so that the four k a wavefront loads per step share their tap; without it (a first layer
// of three channels) in the filter's own order c, r, s, the taps looked up per k.  POINTWISE and C4 test the reduction's
// end once for a wavefront's four k, so both need C a multiple of 4 (of either convolution of a pair); ANY masks each k
// and takes the rest, one-tap filters among them.
enum { D32_POINTWISE = 0, D32_TAPS_C4 = 1, D32_TAPS_ANY = 2 };

template <int BM, int BN, int WM, int WN, int NS, int U, int AV, int BV, int MODE, bool DUAL>
__global__ __launch_bounds__(256) void conv_f32_dma_kernel(const IgemmArgs a, const Dma32Plan pl, float *partials, unsigned *counters) {
#if __HIP_DEVICE_COMPILE__
  static_assert(WM * WN == 4 && BM % (32 * WM) == 0 && BN % (32 * WN) == 0, "four wavefronts over the tile");
  static_assert(BV == 1 || MODE == D32_POINTWISE, "four pixels per lane only without taps");
  constexpr int BK = D32_BK, TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int SUB = BK * (BM + BN) * 4;  // bytes of 16 k; a stage is U of them
  // a wavefront loads rows 4 * wave .. + 3 of both operands; per operand RPI rows per instruction or IPR instructions per row
  constexpr int A_RPI = 64 * AV / BM > 1 ? 64 * AV / BM : 1, A_IPR = BM / (64 * AV) > 1 ? BM / (64 * AV) : 1;
  constexpr int B_RPI = 64 * BV / BN > 1 ? 64 * BV / BN : 1, B_IPR = BN / (64 * BV) > 1 ? BN / (64 * BV) : 1;
  static_assert(A_RPI <= 4 && B_RPI <= 4, "an instruction's rows belong to one wavefront");
  constexpr int L = 4 * A_IPR / A_RPI + 4 * B_IPR / B_RPI;  // loads per wavefront and step
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  // The arguments, all at once: read where they are first used, they came in four rounds in front of the first load and in more at
  // the end, a fraction of a microsecond each: 64 -> 64 at 90x117, 33 layers of it, 662 -> 650 us.  (In registers from the start, as in
  // igemm_f32_small.hip, sizes packed and the plan computed from them: 150 more instructions, no gain.)
  asm volatile("" ::"s"(pl.tiles_m), "s"(pl.whole), "s"(pl.rest), "s"(pl.splits), "s"(pl.round), "s"(pl.units), "s"(pl.steps), "s"(pl.steps_per_split),
               "s"((int)pl.neighbours), "s"(pl.magic_tiles_m), "s"(pl.magic_round), "s"(a.A), "s"(a.X), "s"(a.a_ld), "s"(a.M), "s"(a.Kdim), "s"(a.Ncols),
               "s"(a.H), "s"(a.W), "s"(a.P), "s"(a.Q), "s"(a.sh), "s"(a.sw), "s"(a.x_img_stride), "s"(a.magic_pq), "s"(a.magic_q), "s"(a.bias));
  asm volatile("" ::"s"(a.Y), "s"(a.Cin), "s"(a.y_img_stride), "s"(a.y_row_stride), "s"(a.c_row_stride), "s"(a.act), "s"(a.act_coef), "s"(partials),
               "s"(counters));
  if constexpr (MODE != D32_POINTWISE) asm volatile("" ::"s"(a.R), "s"(a.S), "s"(a.ph), "s"(a.pw));
  if constexpr (DUAL) asm volatile("" ::"s"(a.A2), "s"(a.X2), "s"(a.bias2), "s"(a.Kdim2), "s"(a.H2), "s"(a.W2), "s"(a.sh2), "s"(a.sw2), "s"(a.x2_img_stride));

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int wm0 = (wave / WN) * (BM / WM), wn0 = (wave % WN) * (BN / WN);

  // ---- which tile, which steps --------------------------------------------
  int tile, split = 0, s_beg = 0, s_end = pl.steps;
  const int b = (int)blockIdx.x;
  const bool part = b < pl.units;
  if (part) {
    split = div_magic(b, pl.round, pl.magic_round);
    if (split >= pl.splits) return;
    tile = pl.neighbours ? xcd_tile(b - split * pl.round, pl.rest) : b - split * pl.round;
    if (tile < 0) return;
    tile += pl.whole;
    s_beg = split * pl.steps_per_split;
    s_end = min(s_end, s_beg + pl.steps_per_split);
  } else {  // consecutive tiles (the filter rows of one column range first) on one XCD: they share operands in its L2
    const int w = b - pl.units, per_xcd = (pl.whole + 7) >> 3;
    tile = (w & 7) * per_xcd + (w >> 3);
    if ((w >> 3) >= per_xcd || tile >= pl.whole) return;
  }
  const int tile_n = div_magic(tile, pl.tiles_m, pl.magic_tiles_m), tile_m = tile - tile_n * pl.tiles_m;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int PQ = a.P * a.Q, HW = a.H * a.W, RS = a.R * a.S;
  const int C = MODE == D32_POINTWISE ? a.Kdim : a.Kdim / RS;
  const int Kall = DUAL ? a.Kdim + a.Kdim2 : a.Kdim;

  float bias_mine = 0.f;
  if (a.bias) bias_mine = a.bias[min(m0 + (tid < BM ? tid : 0), a.M - 1)];
  if constexpr (DUAL) {
    if (a.bias2) bias_mine += a.bias2[min(m0 + (tid < BM ? tid : 0), a.M - 1)];
  }

  const int lda4 = 4 * (int)a.a_ld;  // bytes between consecutive k of the filter
  __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.A), 0, (int)(a.Kdim * lda4), 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(a.X), 0, (int)(4 * div_magic(a.Ncols, PQ, a.magic_pq) * a.x_img_stride), 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc_a2 = rsrc_a, rsrc_x2 = rsrc_x;
  if constexpr (DUAL) {
    rsrc_a2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.A2), 0, (int)(a.Kdim2 * lda4), 0x00020000);
    rsrc_x2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.X2), 0, (int)(4 * div_magic(a.Ncols, PQ, a.magic_pq) * a.x2_img_stride), 0x00020000);
  }

  // ---- loader constants: byte offsets of this lane ------------------------
  // rows of one instruction: lane / (64 / RPI); bytes between the rows of a tap: channel to channel
  const int a_step4 = MODE == D32_TAPS_C4 ? lda4 * RS : lda4;
  unsigned a_off[A_IPR];
#pragma unroll
  for (int i = 0; i < A_IPR; i++) {
    const int sub = lane / (64 / A_RPI), m = m0 + AV * (lane % (64 / A_RPI)) + 64 * AV * i;
    a_off[i] = m < a.M ? (unsigned)(sub * a_step4 + 4 * m) : D32_OUT_OF_RANGE;
  }
  int b_off[B_IPR];
  [[maybe_unused]] unsigned b_off2[DUAL ? B_IPR : 1];
  [[maybe_unused]] unsigned out_r[B_IPR], out_s[B_IPR];  // bit r (s): row (column) r (s) of the filter lies outside the image
#pragma unroll
  for (int i = 0; i < B_IPR; i++) {
    const int sub = lane / (64 / B_RPI), col = n0 + BV * (lane % (64 / B_RPI)) + 64 * BV * i;
    const bool ok = col < a.Ncols;
    const int img = ok ? div_magic(col, PQ, a.magic_pq) : 0, pq = ok ? col - img * PQ : 0;
    const int p = div_magic(pq, a.Q, a.magic_q), q = pq - p * a.Q;
    const int ih0 = p * a.sh - a.ph, iw0 = q * a.sw - a.pw;
    b_off[i] = 4 * (img * (int)a.x_img_stride + ih0 * a.W + iw0 + sub * HW);
    if constexpr (DUAL) b_off2[i] = ok ? 4u * (unsigned)(img * (int)a.x2_img_stride + p * a.sh2 * a.W2 + q * a.sw2 + sub * a.H2 * a.W2) : D32_OUT_OF_RANGE;
    if constexpr (MODE == D32_POINTWISE) {
      if (!ok) b_off[i] = (int)D32_OUT_OF_RANGE;
    } else {
      // bits lo .. hi - 1 of the filter's rows are inside
      auto outside = [&](int i0, int extent, int n) -> unsigned {
        const int lo = max(0, -i0), hi = min(n, extent - i0);
        const unsigned below_hi = hi >= 32 ? ~0u : (1u << max(hi, 0)) - 1u, below_lo = lo >= 32 ? ~0u : (1u << lo) - 1u;
        return ok ? ~(below_hi & ~below_lo) : ~0u;
      };
      out_r[i] = outside(ih0, a.H, a.R);
      out_s[i] = outside(iw0, a.W, a.S);
    }
  }

  // ---- cursor of the next step to load (scalar) ---------------------------
  // This wavefront's four k of a step share their tap (TAPS_ANY apart), so a load costs a scalar addition: a_v / b_v are
  // the lane's offsets for the tap, a_s / b_s the scalar ones of the first k, advanced by a_inc / b_inc per step.
  int l_k = s_beg * BK + 4 * wave;
  int l_sub = 0;
  const int b_step4 = 4 * HW;
  unsigned a_v[A_IPR], b_v[B_IPR];
  int a_s = 0, b_s = 0, a_row4 = a_step4, b_row4 = b_step4;
  [[maybe_unused]] int l_c = 0, l_r = 0, l_s = 0, l_end = Kall;
  auto past_the_end = [&]() {  // rows past the reduction's end are zeros
#pragma unroll
    for (int j = 0; j < A_IPR; j++) a_v[j] = D32_OUT_OF_RANGE;
#pragma unroll
    for (int j = 0; j < B_IPR; j++) b_v[j] = D32_OUT_OF_RANGE;
    a_s = b_s = a_row4 = b_row4 = 0;
  };
  auto set_tap = [&]() {  // TAPS_C4: at the start of a run of channels
    if (l_r == a.R) { past_the_end(); return; }
    a_s = (l_c * RS + l_r * a.S + l_s) * lda4;
    b_s = l_c * b_step4;
    const int x_tap = 4 * (l_r * a.W + l_s);
#pragma unroll
    for (int j = 0; j < B_IPR; j++) b_v[j] = (unsigned)(b_off[j] + x_tap) | (((out_r[j] >> l_r) | (out_s[j] >> l_s)) << 31);
  };
  auto set_second = [&]() {  // DUAL: the second convolution's channels
    rsrc_a = rsrc_a2; rsrc_x = rsrc_x2;
#pragma unroll
    for (int j = 0; j < B_IPR; j++) b_v[j] = b_off2[DUAL ? j : 0];
    b_row4 = 4 * a.H2 * a.W2;
    a_s = (l_k - a.Kdim) * lda4;
    b_s = (l_k - a.Kdim) * b_row4;
    l_end = Kall;
  };
#pragma unroll
  for (int j = 0; j < A_IPR; j++) a_v[j] = a_off[j];
  if constexpr (MODE == D32_TAPS_C4) {
    const int tap = l_k / C;
    l_c = l_k - tap * C;
    l_r = tap / a.S;
    l_s = tap - l_r * a.S;
    if (tap >= RS) l_r = a.R;
    set_tap();
  } else if constexpr (MODE == D32_POINTWISE) {
#pragma unroll
    for (int j = 0; j < B_IPR; j++) b_v[j] = (unsigned)b_off[j];
    a_s = l_k * lda4;
    b_s = l_k * b_step4;
    if (DUAL) l_end = a.Kdim;
    if (DUAL && l_k >= a.Kdim) set_second();
    if (l_k >= l_end) past_the_end();
  }
  // Row l_k + i of the step, i = 0 .. 3: its loads, into sub-stage l_sub.
  auto issue_row = [&](auto row_c) {
    constexpr int i = decltype(row_c)::value;
    char *As = smem + l_sub * SUB + (4 * wave + i) * BM * 4, *Bs = smem + l_sub * SUB + BK * BM * 4 + (4 * wave + i) * BN * 4;
    if constexpr (MODE != D32_TAPS_ANY) {
      if constexpr (i % A_RPI == 0)
#pragma unroll
        for (int j = 0; j < A_IPR; j++) d32_load<4 * AV>(rsrc_a, (lds_ptr)(As + 256 * AV * j), a_v[j], a_s + i * a_row4);
      if constexpr (i % B_RPI == 0)
#pragma unroll
        for (int j = 0; j < B_IPR; j++) d32_load<4 * BV>(rsrc_x, (lds_ptr)(Bs + 256 * BV * j), b_v[j], b_s + i * b_row4);
    } else {
      const int k = l_k + i;
      const bool in = k < Kall;
      const int c = div_magic(k, RS, a.magic_rs), tap = k - c * RS, r = div_magic(tap, a.S, a.magic_s), s = tap - r * a.S;
      if constexpr (i % A_RPI == 0) {
        const unsigned past = k + lane / (64 / A_RPI) < Kall ? 0u : D32_OUT_OF_RANGE;  // the reduction may end inside an instruction's rows
#pragma unroll
        for (int j = 0; j < A_IPR; j++) d32_load<4 * AV>(rsrc_a, (lds_ptr)(As + 256 * AV * j), a_v[j] | past, in ? k * lda4 : 0);
      }
      const int x_tap = 4 * (r * a.W + s);
#pragma unroll
      for (int j = 0; j < B_IPR; j++) {
        const unsigned voff = (unsigned)(b_off[j] + x_tap) | (((out_r[j] >> r) | (out_s[j] >> s)) << 31) | (in ? 0u : D32_OUT_OF_RANGE);
        d32_load<4 * BV>(rsrc_x, (lds_ptr)(Bs + 256 * BV * j), voff, in ? c * b_step4 : 0);
      }
    }
  };
  auto advance_loader = [&]() {
    l_sub = l_sub + 1 == NS * U ? 0 : l_sub + 1;
    l_k += BK;
    if constexpr (MODE == D32_TAPS_C4) {
      l_c += BK;
      a_s += BK * a_row4;
      b_s += BK * b_row4;
      if (l_c >= C) {
        while (l_c >= C && l_r < a.R) {  // fewer than 16 channels: more than once
          l_c -= C;
          l_s++;
          if (l_s == a.S) { l_s = 0; l_r++; }
        }
        set_tap();
      }
    } else if constexpr (MODE == D32_POINTWISE) {
      a_s += BK * a_row4;
      b_s += BK * b_row4;
      if (l_k >= l_end) {
        if (DUAL && l_end == a.Kdim) set_second();
        if (l_k >= l_end) past_the_end();
      }
    }
  };
  auto issue_stage = [&]() {
#pragma unroll
    for (int u = 0; u < U; u++) {
      issue_row(std::integral_constant<int, 0>{});
      issue_row(std::integral_constant<int, 1>{});
      issue_row(std::integral_constant<int, 2>{});
      issue_row(std::integral_constant<int, 3>{});
      advance_loader();
    }
  };

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  // The counted waits below assume that the bias is older than every ring load.
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  // ---- the ring ------------------------------------------------------------
  // 16 k are two groups of four MFMA k-pairs; a group's operands are read while the group before is multiplied, loads sit
  // between MFMAs, and the barrier that ends a stage has two MFMAs in front of it still running and two behind it.
  // (One workgroup per compute unit, 64x64 tile, microseconds per 16 k; 0.213 is the matrix pipe alone: 0.41 with offsets
  // and masks computed per load, 0.32 with them per tap, 0.295 with the MFMAs around the barrier, 0.27 with a barrier
  // per 32 k.  Deeper rings and a second accumulator for the dependent chain changed nothing.)
  typedef float floatA __attribute__((ext_vector_type(TM)));
  typedef float floatB __attribute__((ext_vector_type(TN)));
  const unsigned ld_a = (unsigned)(4 * (half * BM + wm0 + TM * l32)), ld_b = (unsigned)(4 * (BK * BM + half * BN + wn0 + TN * l32));
  float fa[2][4][TM], fb[2][4][TN];
  auto read_group = [&](const char *stage, auto slot_c, auto g_c) {
    constexpr int slot = decltype(slot_c)::value, g = decltype(g_c)::value;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const char *pa = stage + ld_a + (4 * g + u) * 2 * BM * 4, *pb = stage + ld_b + (4 * g + u) * 2 * BN * 4;
      if constexpr (TM == 1) fa[slot][u][0] = *reinterpret_cast<const float *>(pa);
      else {
        const floatA v = *reinterpret_cast<const floatA *>(pa);
#pragma unroll
        for (int i = 0; i < TM; i++) fa[slot][u][i] = v[i];
      }
      if constexpr (TN == 1) fb[slot][u][0] = *reinterpret_cast<const float *>(pb);
      else {
        const floatB v = *reinterpret_cast<const floatB *>(pb);
#pragma unroll
        for (int j = 0; j < TN; j++) fb[slot][u][j] = v[j];
      }
    }
  };
  auto mfma_pair = [&](auto slot_c, auto u_c) {
    constexpr int slot = decltype(slot_c)::value, u = decltype(u_c)::value;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[slot][u][i], fb[slot][u][j], acc[i][j], 0, 0, 0);
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 2> c2{};
  constexpr std::integral_constant<int, 3> c3{};
  constexpr int P = NS - 1;  // stages in flight behind the one being computed
  static_assert(P >= 1 && P <= 4 && (P - 1) * L * U < 64, "ring depth");
  int c_stage = 0;
#define PIN() __builtin_amdgcn_sched_barrier(0)
  auto stage_body = [&](auto g_c, auto loads_c) {
    constexpr int G = decltype(g_c)::value;  // stages still in flight when this one ends
    constexpr bool LOADS = decltype(loads_c)::value;
    const char *stage = smem + c_stage * (U * SUB);
    c_stage = c_stage + 1 == NS ? 0 : c_stage + 1;
#pragma unroll
    for (int u = 0; u < U; u++) {
      mfma_pair(c0, c0); PIN();
      read_group(stage + u * SUB, c1, c1); PIN();  // behind an MFMA: the wait for the group before covers nothing newer
      if constexpr (LOADS) { issue_row(c0); PIN(); }
      mfma_pair(c0, c1); PIN();
      if constexpr (LOADS) { issue_row(c1); PIN(); }
      mfma_pair(c0, c2); PIN();
      if constexpr (LOADS) { issue_row(c2); PIN(); }
      mfma_pair(c0, c3); PIN();
      if constexpr (LOADS) { issue_row(c3); advance_loader(); PIN(); }
      mfma_pair(c1, c0); mfma_pair(c1, c1); PIN();
      if (u + 1 < U) {
        read_group(stage + (u + 1) * SUB, c0, c0); PIN();
      } else if constexpr (G > 0) {
        // The pipe still works through the MFMAs above.  This wavefront's part of the next stage has landed and its
        // reads of this one are done (lgkmcnt 0); behind the barrier that holds for all four, and the loads issued
        // during the next stage may overwrite this one.
        d32_wait_vmcnt<(G - 1) * L * U, 0>();
        d32_barrier();
        read_group(smem + c_stage * (U * SUB), c0, c0); PIN();
      }
      mfma_pair(c1, c2); mfma_pair(c1, c3); PIN();
    }
  };
  const int nk = (s_end - s_beg + U - 1) / U;  // a last stage that is not full loads zeros
  {
    const int pre = nk < P ? nk : P;
#pragma unroll
    for (int q = 0; q < P; q++)
      if (q < pre) issue_stage();
    if (pre == 1) d32_wait_vmcnt<0>();
    else if (pre == 2) d32_wait_vmcnt<(P > 1 ? 1 : 0) * L * U>();
    else if (pre == 3) d32_wait_vmcnt<(P > 2 ? 2 : 0) * L * U>();
    else d32_wait_vmcnt<(P > 3 ? 3 : 0) * L * U>();
    d32_barrier();
    read_group(smem, c0, c0); PIN();
  }
  for (int it = 0; it < nk - P; it++) stage_body(std::integral_constant<int, P>{}, std::true_type{});
  if constexpr (P > 3) { if (nk > 3) stage_body(std::integral_constant<int, 3>{}, std::false_type{}); }
  if constexpr (P > 2) { if (nk > 2) stage_body(std::integral_constant<int, 2>{}, std::false_type{}); }
  if constexpr (P > 1) { if (nk > 1) stage_body(std::integral_constant<int, 1>{}, std::false_type{}); }
  stage_body(std::integral_constant<int, 0>{}, std::false_type{});
#undef PIN

  d32_barrier();  // nobody reads the operand stages any more
  float *bias_s = reinterpret_cast<float *>(smem);                          // [BM]
  volatile unsigned *arrived_s = reinterpret_cast<unsigned *>(smem + BM * 4);

  // ---- a split tile: the hand-over of the other fp32 kernels (igemm_f32_small.hip states what it rests on) ----
  if (part && pl.splits > 1) {
    constexpr int TILE = BM * BN;
    const int rt = tile - pl.whole;
    const __amdgpu_buffer_rsrc_t parts = part_rsrc(partials);
    const unsigned mine = 16u * (unsigned)tid, first_part = (unsigned)(rt * pl.splits) * (4u * TILE);  // [four registers][thread]
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const floatx16 &o = acc[i][j];
          part_store(parts, mine + 4096 * ((i * TN + j) * 4 + g), first_part + (unsigned)split * (4u * TILE), part_floatx4{o[4 * g], o[4 * g + 1], o[4 * g + 2], o[4 * g + 3]});
        }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (tid == 0) *arrived_s = __hip_atomic_fetch_add(&counters[rt], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived_s != (unsigned)pl.splits - 1) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    constexpr int AT_ONCE = 4 / (TM * TN);  // no more registers than the reduction leaves free
    for (int y = 0; y < pl.splits; y += AT_ONCE) {  // so many parts in flight, added in split order
      part_floatx4 p[AT_ONCE][TM * TN * 4];
#pragma unroll
      for (int u = 0; u < AT_ONCE; u++)
#pragma unroll
        for (int g = 0; g < TM * TN * 4; g++)
          p[u][g] = part_load<part_floatx4>(parts, y + u < pl.splits ? mine + 4096 * g : PART_NONE, first_part + (unsigned)min(y + u, pl.splits - 1) * (4u * TILE));
#pragma unroll
      for (int u = 0; u < AT_ONCE; u++)
#pragma unroll
        for (int g = 0; g < TM * TN * 4; g++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[g / 4 / TN][g / 4 % TN][4 * (g & 3) + e] += p[u][g][e];
    }
    if (tid == 0) __hip_atomic_store(&counters[rt], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // ---- epilogue: (acc + bias) + residual, activation ------------------------
  // register r of block (i, j): k_out m0 + wm0 + TM * (8 * (r / 4) + 4 * half + r % 4) + i, pixel n0 + wn0 + TN * l32 + j
  if (tid < BM) bias_s[tid] = bias_mine;
  __syncthreads();
  const int col = n0 + wn0 + TN * l32;
  const bool ok0 = col < a.Ncols, ok1 = TN > 1 && col + 1 < a.Ncols;
  const int colc = ok0 ? col : 0;
  const int img = div_magic(colc, PQ, a.magic_pq), pq = colc - img * PQ;
  const int64_t at0 = (int64_t)img * a.y_img_stride + pq;
  const int64_t at1 = pq + 1 < PQ ? at0 + 1 : (int64_t)(img + 1) * a.y_img_stride;  // the lane's second pixel, in the next image now and then
  const bool pairs = TN > 1 && __all(ok1 && pq + 1 < PQ);  // every lane's two pixels are neighbours in memory
  const int mrow = m0 + wm0 + TM * 4 * half;               // + TM * (8 * (r >> 2) + (r & 3)) + i
  float *__restrict__ Yg = a.Y + (int64_t)mrow * a.y_row_stride;
  const float *__restrict__ Cg = a.Cin ? a.Cin + (int64_t)mrow * a.c_row_stride : nullptr;
  const bool full = m0 + BM <= a.M;
  auto finish = [&](auto mode_c, auto full_c, auto pair_c) {
    constexpr int ACT = decltype(mode_c)::value;
    constexpr bool FULL = decltype(full_c)::value, PAIR = decltype(pair_c)::value;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      float z0[16], z1[16];
      if (Cg) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int k = TM * (8 * (r >> 2) + (r & 3)) + i;
          const int64_t o = (int64_t)(FULL ? k : min(k, a.M - 1 - mrow)) * a.c_row_stride;
          if constexpr (PAIR) {
            const float2u v = *reinterpret_cast<const float2u *>(Cg + at0 + o);
            z0[r] = v[0]; z1[r] = v[1];
          } else {
            z0[r] = Cg[at0 + o];
            if constexpr (TN > 1) z1[r] = Cg[(ok1 ? at1 : at0) + o];
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int k = TM * (8 * (r >> 2) + (r & 3)) + i;
        if (!FULL && mrow + k >= a.M) continue;
        const float bv = bias_s[wm0 + TM * 4 * half + k];
        float v0 = acc[i][0][r] + bv, v1 = TN > 1 ? acc[i][TN - 1][r] + bv : 0.f;
        if (Cg) { v0 += z0[r]; if (TN > 1) v1 += z1[r]; }
        v0 = apply_act(v0, ACT, a.act_coef);
        v1 = apply_act(v1, ACT, a.act_coef);
        const int64_t o = (int64_t)k * a.y_row_stride;
        if constexpr (PAIR) {
          const float2u v = {v0, v1};
          *reinterpret_cast<float2u *>(Yg + at0 + o) = v;
        } else {
          if (ok0) Yg[at0 + o] = v0;
          if (ok1) Yg[at1 + o] = v1;
        }
      }
    }
  };
  auto finish_mode = [&](auto mode_c) {
    if (!full) finish(mode_c, std::false_type{}, std::false_type{});
    else if (pairs) finish(mode_c, std::true_type{}, std::integral_constant<bool, (TN > 1)>{});
    else finish(mode_c, std::true_type{}, std::false_type{});
  };
  switch (a.act) {
    case DNNRT_ACT_RELU: finish_mode(std::integral_constant<int, DNNRT_ACT_RELU>{}); break;
    case DNNRT_ACT_CLIPPED_RELU: finish_mode(std::integral_constant<int, DNNRT_ACT_CLIPPED_RELU>{}); break;
    case DNNRT_ACT_LEAKY_RELU: finish_mode(std::integral_constant<int, DNNRT_ACT_LEAKY_RELU>{}); break;
    default: finish_mode(std::integral_constant<int, DNNRT_ACT_IDENTITY>{}); break;
  }
#endif
}

template <int BM, int BN, int WM, int WN, int NS, int U, int AV, int BV, int MODE, bool DUAL>
static bool launch_one(const dnnrtContext *ctx, const IgemmArgs &a, const Dma32Plan &pl) {
  constexpr int SMEM = NS * U * D32_BK * (BM + BN) * 4;
  static_assert(SMEM <= 64 * 1024, "no more LDS than a kernel gets without asking");
  const unsigned grid = (unsigned)(pl.units + ceil_div(pl.whole, 8) * 8);
  hipLaunchKernelGGL((conv_f32_dma_kernel<BM, BN, WM, WN, NS, U, AV, BV, MODE, DUAL>), dim3(grid), dim3(256), SMEM, ctx->stream, a, pl,
                     ctx->splitk_partials, ctx->splitk_counters);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("conv(fp32, dma): launch failed: %s", hipGetErrorString(e)); return false; }
  return true;
}

template <int BM, int BN, int WM, int WN, int NS, int U>
static bool launch_tile32(const dnnrtContext *ctx, const IgemmArgs &a, const Dma32Plan &pl, int mode, bool av4, bool bv4) {
  constexpr int AV = BM >= 64 ? 4 : 1;
  const bool dual = a.A2 != nullptr;
#define D32(AV_, BV_, MODE_, DUAL_) return launch_one<BM, BN, WM, WN, NS, U, AV_, BV_, MODE_, DUAL_>(ctx, a, pl)
  if (dual) {
    if constexpr (BM >= 64) {
      if (bv4) D32(AV, 4, D32_POINTWISE, true);
      D32(AV, 1, D32_POINTWISE, true);
    }
    return false;
  }
  if (mode == D32_POINTWISE) {
    if (av4 && bv4) D32(AV, 4, D32_POINTWISE, false);
    if (av4) D32(AV, 1, D32_POINTWISE, false);
    D32(1, 1, D32_POINTWISE, false);
  }
  if (mode == D32_TAPS_C4) {
    if (av4) D32(AV, 1, D32_TAPS_C4, false);
    D32(1, 1, D32_TAPS_C4, false);
  }
  if (av4) D32(AV, 1, D32_TAPS_ANY, false);
  D32(1, 1, D32_TAPS_ANY, false);
#undef D32
}

bool launch_conv_f32_dma(const dnnrtContext *ctx, const IgemmArgs &args, double at_most_us, bool &launched) {
  launched = false;
  IgemmArgs a = args;
  const bool dual = a.A2 != nullptr;
  const int PQ = a.P * a.Q;
  const int64_t images = a.Ncols / PQ;
  const int64_t lim = (1ll << 31) - 4096;
  if (!a.a_mcontig || a.b_kcontig || a.Z != 1 || a.bias_col || a.alpha != 1.f || (a.Cin && a.beta != 1.f) || a.act == ACT_GELU || a.R > 32 || a.S > 32 ||
      images * PQ != a.Ncols || a.x_img_stride < (int64_t)(a.Kdim / (a.R * a.S)) * a.H * a.W || 4 * images * a.x_img_stride > lim || 4 * (int64_t)a.Kdim * a.a_ld > lim)
    return true;
  const bool pointwise = a.R == 1 && a.S == 1 && a.ph == 0 && a.pw == 0;
  if (dual && (!pointwise || a.Kdim % 4 || a.Kdim2 % 4 || 4 * images * a.x2_img_stride > lim || 4 * (int64_t)a.Kdim2 * a.a_ld > lim)) return true;
  const int RS = a.R * a.S, C = a.Kdim / RS;
  const bool av4 = a.M % 4 == 0 && a.a_ld % 4 == 0 && aligned16(a.A) && (!dual || aligned16(a.A2));
  if (dual && !av4) return true;
  const bool bv4 = pointwise && a.sh == 1 && a.sw == 1 && PQ % 4 == 0 && C % 4 == 0 && aligned16(a.X) &&
                   (!dual || (a.sh2 == 1 && a.sw2 == 1 && aligned16(a.X2)));
  const int mode = C % 4 ? D32_TAPS_ANY : pointwise ? D32_POINTWISE : D32_TAPS_C4;
  a.magic_pq = magic_of(PQ);
  a.magic_q = magic_of(a.Q);
  a.magic_rs = magic_of(RS);
  a.magic_s = magic_of(a.S);

  // Estimated time of each tile shape and split depth, in microseconds (measured on layers of 0.1 .. 60 GFLOP): a
  // compute unit with one workgroup takes t1 per step of 16 k, one with several takes tm per workgroup and step; launch,
  // first data and stores are 4 to 5, a split tile's hand-over 3 and the reading of its parts.
  static const struct { int bm, bn; double t1, tm; } shapes[] = {
      {128, 128, 0.96, 0.90}, {64, 128, 0.52, 0.46}, {128, 64, 0.51, 0.46}, {64, 64, 0.27, 0.242}, {32, 128, 0.29, 0.26}};
  const int steps = (int)ceil_div((dual ? a.Kdim + a.Kdim2 : a.Kdim), D32_BK);
  int best_shape = -1;
  double best = 0;
  Dma32Plan pl{};
  for (int i = 0; i < 5; i++) {
    const int bm = shapes[i].bm, bn = shapes[i].bn;
    if (dual && bm < 64) continue;
    const int64_t tiles = ceil_div(a.M, bm) * ceil_div(a.Ncols, bn);
    if (tiles > (1 << 28)) continue;
    const double fixed = pointwise ? 4.0 : 5.0;
    const int64_t rounds = tiles / ctx->num_cu, rest = tiles - rounds * ctx->num_cu;
    for (int s = 1; s <= 16; s++) {
      if (s > 1 && (rest == 0 || ctx->splitk_shared || steps / s < 2 || rest * s * bm * bn * 4 > ctx->splitk_partial_bytes || rest > ctx->splitk_max_tiles)) break;
      const int unit = bm * bn <= 4096 ? 2 : 1;  // 16-k steps per ring stage: a part starts on a stage
      const int per = (int)ceil_div(ceil_div(steps, s), unit) * unit;
      if (ceil_div(steps, per) != s) continue;
      // Parts of neighbouring tiles on one XCD, or every eighth tile (with the usual multiples of eight filter-row tiles:
      // one range of filters per XCD): whichever operand is the larger is fetched once, the other by all eight L2s.  The
      // activations count once a tap, as a tap's pass over the channels outlasts what an L2 keeps.  512 -> 512, 3x3
      // stride 2 at 14x14, batch 32: 119 -> 84 us, 256 -> 256 at 28x28: 79 -> 72.  A tile's parts stay on one XCD
      // and consecutive workgroups are of different tiles: the other way round layers of few tiles lost 10 to 20%.
      const bool neighbours = (rest % 8 == 0 || rest >= 64) && (int64_t)a.M * a.Kdim <= images * a.x_img_stride * RS;
      const int64_t parts = neighbours ? ceil_div(ceil_div(rest, 8) * s, ceil_div(ctx->num_cu, 8)) : ceil_div(rest * s, ctx->num_cu);  // of a split tile, on the busiest compute unit
      const double load = (double)rounds * steps + (double)parts * per;
      double cost = load * (rounds + parts > 1 ? shapes[i].tm : shapes[i].t1) + fixed;
      if (rounds + parts > 1 && cost < fixed + shapes[i].t1 * per) cost = fixed + shapes[i].t1 * per;
      if (s > 1) cost += (rounds > 0 ? 2.5 : 3.0) + s * (bm * bn / 4096.0) * 0.3;  // partly behind the whole tiles
      if (best_shape < 0 || cost < best) {
        best = cost;
        best_shape = i;
        pl.tiles_m = (int)ceil_div(a.M, bm);
        pl.splits = s;
        pl.rest = s > 1 ? (int)rest : 0;
        pl.whole = (int)tiles - pl.rest;
        pl.neighbours = s > 1 && neighbours;
        pl.round = pl.neighbours ? (int)ceil_div(pl.rest, 8) * 8 : pl.rest;
        pl.units = (int)(ceil_div((int64_t)pl.round * s, 8) * 8);
        pl.steps = steps;
        pl.steps_per_split = per;
      }
    }
  }
  // 3x3 layers with stride 1: by Winograd's method where that is estimated to be faster and the caller has not asked for direct sums
  if (!a.direct_sums && !launch_conv_f32_winograd(ctx, args, best_shape < 0 || best > at_most_us ? at_most_us : best, launched)) return false;
  if (launched) return true;
  if (best_shape < 0 || best > at_most_us) return true;
  pl.magic_tiles_m = magic_of(pl.tiles_m);
  pl.magic_round = magic_of(pl.round > 0 ? pl.round : 1);
  launched = true;
  switch (best_shape) {
    case 0: return launch_tile32<128, 128, 2, 2, 3, 1>(ctx, a, pl, mode, av4, bv4);
    case 1: return launch_tile32<64, 128, 2, 2, 4, 1>(ctx, a, pl, mode, av4, bv4);
    case 2: return launch_tile32<128, 64, 2, 2, 4, 1>(ctx, a, pl, mode, av4, bv4);
    case 3: return launch_tile32<64, 64, 2, 2, 3, 2>(ctx, a, pl, mode, av4, bv4);
    default: return launch_tile32<32, 128, 1, 4, 3, 2>(ctx, a, pl, mode, av4, bv4);
  }
}

}  // namespace dnnrt
