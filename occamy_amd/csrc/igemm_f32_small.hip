// Two specialisations of the small-problem fp32 implicit GEMM
// (igemm_f32_direct.hip) for the shapes that make up a batch-1 CNN or a short
// transformer: 3x3 convolutions and 1x1 convolutions / plain matrix products.
//
// Same decomposition -- one 32x32 tile of D per workgroup, KS wavefronts
// splitting the reduction, operands straight from global memory into MFMA
// registers -- but the per-element index arithmetic is gone (a wave64 VALU
// instruction costs 4 cycles, and ~30 of them per loaded element made the
// general kernel issue-bound):
//   3x3: a lane owns one output pixel; its nine tap offsets and nine validity
//        masks are computed once.  One iteration = 2 channels x 9 taps
//        (half-wave h takes channel c+h), i.e. nine MFMAs fed by nine
//        contiguous filter words and nine input words at base + tap_off[j].
//   1x1: the reduction index is the channel; addresses advance by a constant.
// All loads go to the lane's offset plus a scalar one, what must not contribute has bit 31 of its offset set and reads zero: no
// vector instruction per load and none per MFMA (there were two and two; conv 3x3 64 -> 64 at 56x56 8.0 -> 7.7 us, with the
// work behind the reduction spread over the wavefronts; ResNet-50 at batch 1 423 -> 400).  The compiler can track the
// hardware load counter and the register ring keeps several iterations of
// loads in flight.  Offsets are 31-bit: the dispatcher only takes these
// kernels when every operand is below 2^29 elements.
#include "igemm_f32.h"
#include "partials.h"

#include <type_traits>

namespace dnnrt {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// Operands are read with raw buffer loads: the lane's offset and a scalar one, so a load costs no vector instruction (an fp32
// MFMA and the vector instructions share their multipliers: they take turns).  A lane whose offset has bit 31 set reads zero.
[[maybe_unused]] constexpr unsigned SMALL_OUT_OF_RANGE = 0x80000000u;
#if __HIP_DEVICE_COMPILE__
__device__ __forceinline__ __amdgpu_buffer_rsrc_t small_rsrc(const float *base) {  // offsets below 2^31 are the caller's care
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ float small_load(__amdgpu_buffer_rsrc_t rsrc, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)voff, (int)soff, 0));
}
typedef unsigned small_uintx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 small_load4(__amdgpu_buffer_rsrc_t rsrc, unsigned voff, unsigned soff) {
  const small_uintx4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)voff, (int)soff, 0);
  return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}
#endif

// The 16 accumulator registers of a lane hold rows m0 + 8 * (r >> 2) + 4 * half + (r & 3)
// of output column n0 + l32.
__device__ __forceinline__ int acc_row(int m0, int half, int r) { return m0 + 8 * (r >> 2) + 4 * half + (r & 3); }
// ... that is, row m0 + 4 * half (the only part that differs between lanes) plus row_k(r), known at compile time:
// address arithmetic per row is then a uniform offset (scalar unit) added to one per-lane base.
__device__ __forceinline__ constexpr int row_k(int r) { return 8 * (r >> 2) + (r & 3); }

// Of a tile's 16 accumulator registers each of the KS wavefronts finishes 16 / KS: what they need beside the sums (bias of
// a register's row, residual of its element), requested at kernel start so that the values are there when the epilogue wants them.
template <int KS>
struct Finish {
  static constexpr int N = 16 / KS;
  float bias[N], res[N];
};
template <int KS>
__device__ __forceinline__ void prefetch_finish(const IgemmArgs &a, int z, int m0, int half, int wave, int img, int pq, Finish<KS> &f) {
  constexpr int N = Finish<KS>::N;
  const float *__restrict__ biasg = a.bias ? a.bias + (int64_t)z * a.bias_z_stride : nullptr;
  const float *__restrict__ Cg = a.Cin ? a.Cin + (int64_t)z * a.c_z_stride + (int64_t)img * a.y_img_stride + pq : nullptr;
#pragma unroll
  for (int i = 0; i < N; i++) {
    const int row = min(acc_row(m0, half, wave * N + i), a.M - 1);
    f.bias[i] = biasg ? biasg[row] : 0.f;
    f.res[i] = Cg ? Cg[(int64_t)row * a.c_row_stride] : 0.f;
  }
}

// Sum the KS partial tiles in LDS, then bias / residual / activation / store, 16 / KS registers of the tile per wavefront (on one
// wavefront alone the reads of the other seven's sums, and of up to sixteen parts, are a chain of 112 and 256 loads).
// The reduction may also be split over gridDim.y workgroups.  Each of them
// leaves its partial tile in `partials` and bumps the tile's arrival counter;
// whoever arrives last adds the partials up in split order -- the order of
// arrival does not matter, so the result is the same bits on every run -- and
// finishes the tile.  Nobody waits for anybody.  The last arriver puts the
// counter back to zero for the next kernel on the stream.
template <int KS>
__device__ __forceinline__ void reduce_and_store(const IgemmArgs &a, floatx16 acc, const Finish<KS> &f, float bias_c, float (*red)[16][64],
                                                 int wave, int lane, int m0, int img, int pq, bool col_ok, int z, unsigned tile, int splits,
                                                 float *partials, unsigned *counters) {
  constexpr int N = 16 / KS;
  const int half = lane >> 5;
  float v[N];
  if constexpr (KS > 1) {
#pragma unroll
    for (int r = 0; r < 16; r++) red[wave][r][lane] = acc[r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; i++) {
      v[i] = red[0][wave * N + i][lane];
#pragma unroll
      for (int w = 1; w < KS; w++) v[i] += red[w][wave * N + i][lane];
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = acc[i];
  }
  if (splits > 1) {
#if __HIP_DEVICE_COMPILE__
    // a partial tile: [wavefront][vector of its registers][lane]
    typedef std::conditional_t<N == 2, part_floatx2, part_floatx4> vec_t;
    constexpr int E = N == 2 ? 2 : 4, VECS = N / E;
    const __amdgpu_buffer_rsrc_t parts = part_rsrc(partials);
    const unsigned mine = (unsigned)(wave * N * 256 + lane * 4 * E), first_part = tile * (unsigned)splits * 4096u;
#pragma unroll
    for (int i = 0; i < VECS; i++) {
      vec_t o;
#pragma unroll
      for (int e = 0; e < E; e++) o[e] = v[E * i + e];
      part_store(parts, mine + 256 * E * i, first_part + 4096u * blockIdx.y, o);
    }
    // The hand-over.  Every wavefront of every workgroup of a tile (1) writes its part of the partial tile with device-scope
    // stores, which go past the per-XCD L2 to the point where all XCDs agree, (2) waits until every one of
    // them is acknowledged (s_waitcnt 0: the counters of a wavefront reach zero only when its stores have been
    // written there); behind the workgroup's barrier (3) one thread adds one to the tile's arrival counter with a device-scope
    // atomic, performed at that same point.  Whoever reads splits - 1 knows that every other workgroup's step (2) is over, so its
    // device-scope loads, issued after the counter's value has come back (the branch depends on it and
    // a wavefront issues in order), read the finished partial tiles.  Nobody waits for anybody: a workgroup
    // that is not last leaves.  What this rests on is the hardware's behaviour, stated above, not the
    // language's memory model, which would ask for a release on (3) and an acquire in the reader; on this
    // target a release at device scope also writes back every dirty line of the XCD's L2 (the previous
    // layer's output), which costs more than the split saves.  The signal fences keep the compiler, which
    // may reorder relaxed accesses to different addresses, from moving them across (2) and (3); they emit no
    // instruction.
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);  // vmcnt(0) expcnt(0) lgkmcnt(0)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    unsigned arrived = 0;
    if constexpr (KS > 1) {
      __syncthreads();
      volatile unsigned *arrived_s = reinterpret_cast<unsigned *>(&red[0][0][0]);  // the sums have been read
      if (wave == 0 && lane == 0) *arrived_s = __hip_atomic_fetch_add(&counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      arrived = *arrived_s;
    } else if (lane == 0) {
      arrived = __hip_atomic_fetch_add(&counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    arrived = __builtin_amdgcn_readfirstlane(arrived);
    if (arrived != (unsigned)splits - 1) return;
    if (wave == 0 && lane == 0) __hip_atomic_store(&counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the partial tiles are requested as many at a time as there are up to 32 values, and added in split order
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = 0.f;
    auto add_parts = [&](int y, auto at_once_c) {
      constexpr int AT_ONCE = decltype(at_once_c)::value;
      vec_t p[AT_ONCE][VECS];
#pragma unroll
      for (int u = 0; u < AT_ONCE; u++)
#pragma unroll
        for (int i = 0; i < VECS; i++)
          p[u][i] = part_load<vec_t>(parts, y + u < splits ? mine + 256 * E * i : PART_NONE, first_part + 4096u * (unsigned)min(y + u, splits - 1));
#pragma unroll
      for (int u = 0; u < AT_ONCE; u++)
#pragma unroll
        for (int i = 0; i < N; i++) v[i] += p[u][i / E][i % E];
    };
    constexpr int MOST = N <= 2 ? 16 : N == 4 ? 8 : N == 8 ? 4 : 2;
    if (MOST > 4 && splits <= 4) add_parts(0, std::integral_constant<int, 4>{});
    else
      for (int y = 0; y < splits; y += MOST) add_parts(y, std::integral_constant<int, MOST>{});
#endif
  }
  if (!col_ok) return;
  const int row0 = acc_row(m0, half, wave * N);  // the rows of a wavefront's registers: row0 + row_k(wave * N + i) - row_k(wave * N)
  float *__restrict__ y0 = a.Y + (int64_t)z * a.y_z_stride + (int64_t)img * a.y_img_stride + pq;
  // one copy of the store loop per activation mode, picked once (the mode is the same for every lane)
  auto store = [&](auto mode_c) {
    constexpr int MODE = decltype(mode_c)::value;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int row = N <= 4 ? row0 + i : acc_row(m0, half, wave * N + i);  // four registers are four consecutive rows
      if (row >= a.M) continue;
      float x = a.alpha * v[i] + f.bias[i] + bias_c;
      if (a.Cin) x += a.beta * f.res[i];
      y0[(int64_t)row * a.y_row_stride] = apply_act(x, MODE, a.act_coef);
    }
  };
  switch (a.act) {
    case DNNRT_ACT_RELU: store(std::integral_constant<int, DNNRT_ACT_RELU>{}); break;
    case DNNRT_ACT_CLIPPED_RELU: store(std::integral_constant<int, DNNRT_ACT_CLIPPED_RELU>{}); break;
    case DNNRT_ACT_LEAKY_RELU: store(std::integral_constant<int, DNNRT_ACT_LEAKY_RELU>{}); break;
    case ACT_GELU: store(std::integral_constant<int, ACT_GELU>{}); break;
    default: store(std::integral_constant<int, DNNRT_ACT_IDENTITY>{}); break;
  }
}

// The 3x3 kernel's iterations 0 .. niter - 1: load(i, slot, last) and multiply(slot) in a ring of three slots, each loaded two
// ahead of its multiplication; `last` says where i can be the last iteration, which may have only its first half.  A compute unit
// accepts one of these 4-byte loads in six cycles, and an iteration has eighteen a wavefront: with four requested first (most batch-1
// layers have no more a wavefront), 1.7 us passed before the first MFMA.  Two ahead are 1 us of MFMA
// work, which covers the latency: 64 -> 64 at 56x56 7.71 -> 6.75 us, ResNet-50 at batch 1 399 -> 385; and with three slots for four two
// workgroups of eight wavefronts fit a compute unit: 6.5 and 379, 128 -> 128 at 28x28, batch 4, 17.3 -> 15.6.  (The 1x1 kernel's
// iterations are 0.2 us: there four slots stay in flight; two ahead cost MobileNetV2 2%.)  The counted waits
// need code in which it is certain which loads have been issued, hence the groups of three without a branch and the endings.
template <class Load, class Multiply, class Then>
__device__ __forceinline__ void small_pipeline(int niter, Load load, Multiply multiply, Then then) {
  constexpr std::integral_constant<int, 0> s0{};
  constexpr std::integral_constant<int, 1> s1{};
  constexpr std::integral_constant<int, 2> s2{};
  constexpr std::true_type perhaps_last{};
  constexpr std::false_type not_last{};
  if (niter >= 3) {
    load(0, s0, not_last);
    load(1, s1, not_last);
    then();
    int i = 0;
    for (; i + 5 <= niter; i += 3) {
      load(i + 2, s2, not_last); multiply(s0);
      load(i + 3, s0, not_last); multiply(s1);
      load(i + 4, s1, perhaps_last); multiply(s2);
    }
    // two to four are left, the first two of them requested
    if (i + 4 == niter) {
      load(i + 2, s2, not_last); multiply(s0);
      load(i + 3, s0, perhaps_last); multiply(s1);
      multiply(s2);
      multiply(s0);
    } else {
      if (i + 3 == niter) load(i + 2, s2, perhaps_last);
      multiply(s0);
      multiply(s1);
      if (i + 3 == niter) multiply(s2);
    }
    return;
  }
  if (niter > 0) load(0, s0, perhaps_last);
  if (niter > 1) load(1, s1, perhaps_last);
  then();
  if (niter > 0) multiply(s0);
  if (niter > 1) multiply(s1);
}

// The arguments in front of the struct are in registers when a wavefront starts.  PLAIN: they are all that the loads need (one
// image size in and out, stride 1, one z, images side by side, one reduction), and nothing waits for the rest, which comes 0.45 us
// later: ResNet-50 at batch 1, 48 of its 51 launches in these kernels, 379 -> 359 us, 64 -> 64 3x3 at 56x56 6.5 -> 5.8; otherwise only the struct and per_wave are read.  per_wave: the slice of the reduction a wavefront takes, times 4, and log2 of the
// XCD grid's columns.
template <bool PLAIN>
__device__ __forceinline__ IgemmArgs small_args(const float *A, const float *X, int M, int Ncols, int Kdim, int a_ld, int H, int W, int RS, unsigned per_wave,
                                                unsigned magic_tn_per, unsigned magic_pq, const IgemmArgs &args) {
  IgemmArgs a = args;
  if constexpr (PLAIN) {
    a.A = A; a.X = X; a.M = M; a.Ncols = Ncols; a.Kdim = Kdim; a.a_ld = a_ld;
    a.H = a.P = H; a.W = a.Q = W; a.sh = a.sw = 1;
    a.ph = a.pw = RS == 9 ? 1 : 0;
    a.x_img_stride = (int64_t)(Kdim / RS) * (H * W);
    a.xcd_n_log2 = (int)(per_wave & 3);
    a.tm_per = ((M + 31) / 32 + (8 >> a.xcd_n_log2) - 1) >> (3 - a.xcd_n_log2);
    a.tn_per = ((Ncols + 31) / 32 + (1 << a.xcd_n_log2) - 1) >> a.xcd_n_log2;
    a.magic_tn_per = magic_tn_per;
    a.magic_pq = magic_pq;
    a.A2 = nullptr;
    a.a_z_stride = a.x_z_stride = 0;
  } else {  // all at once: read where they are first used, they come in several rounds (the same network 359.5 -> 357.9)
    asm volatile("" ::"s"(a.A), "s"(a.X), "s"(a.M), "s"(a.Ncols), "s"(a.Kdim), "s"(a.a_ld), "s"(a.H), "s"(a.W), "s"(a.P), "s"(a.Q), "s"(a.sh), "s"(a.sw),
                 "s"(a.x_img_stride), "s"(a.a_z_stride), "s"(a.x_z_stride), "s"(a.xcd_n_log2), "s"(a.tm_per), "s"(a.tn_per), "s"(a.magic_tn_per), "s"(a.magic_pq),
                 "s"(a.magic_q), "s"(a.A2), "s"(a.bias), "s"(a.Cin));
    if (RS == 1) asm volatile("" ::"s"(a.X2), "s"(a.Kdim2), "s"(a.H2), "s"(a.W2), "s"(a.sh2), "s"(a.sw2), "s"(a.x2_img_stride), "s"(a.bias2));
  }
  return a;
}
// What the end of the kernel needs, requested at once: read where it is used, each is waited for there.
#define SMALL_LATE_ARGS()                                                                                                                  \
  asm volatile("" : "+s"(a.bias), "+s"(a.bias_col), "+s"(a.Cin), "+s"(a.c_row_stride), "+s"(a.Y), "+s"(a.y_row_stride), "+s"(a.y_img_stride), "+s"(a.alpha), \
               "+s"(a.beta), "+s"(a.act), "+s"(a.act_coef), "+s"(splits), "+s"(partials), "+s"(counters))

template <int KS, bool AMC, bool PLAIN>
__global__ __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(KS >= 2 ? 4 : 3))) void conv3x3_f32_small_kernel(
    const float *A, const float *X, int M, int Ncols, int Kdim, int a_ld, int H, int W, unsigned per_wave, unsigned magic_tn_per, unsigned magic_pq,
    unsigned magic_q, const IgemmArgs args, int splits, float *partials, unsigned *counters) {
  #if __HIP_DEVICE_COMPILE__
  IgemmArgs a = small_args<PLAIN>(A, X, M, Ncols, Kdim, a_ld, H, W, 9, per_wave, magic_tn_per, magic_pq, args);
  if constexpr (PLAIN) a.magic_q = magic_q;
  const int c_per_wave = (int)(per_wave >> 2);
  __shared__ float red[KS > 1 ? KS : 1][16][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, half = lane >> 5;
  // Workgroups go round-robin over the 8 XCDs (gridDim.x is a multiple of 8, so that holds for every y and
  // z as well), each with its own L2.  The XCDs are laid out as a grid of xcd_m x (8 / xcd_m) over the
  // (filter-row tile, column tile) plane and each owns one rectangle of tiles: it fetches 1 / xcd_m of the
  // filter and xcd_m / 8 of the activations, where a run of consecutive tiles per XCD fetches all of one operand
  // into all eight L2s.  The launcher picks xcd_m from the two operands' sizes.
  const int tiles_m = (a.M + 31) / 32, tiles_n = (a.Ncols + 31) / 32, tiles = tiles_n * tiles_m;
  const int tm_per = a.tm_per, tn_per = a.tn_per;
  const int xcd = (int)(blockIdx.x & 7), in_xcd = (int)(blockIdx.x >> 3);
  const int tm_local = div_magic(in_xcd, tn_per, a.magic_tn_per);
  const int tile_m = (xcd >> a.xcd_n_log2) * tm_per + tm_local;
  const int tile_n = (xcd & ((1 << a.xcd_n_log2) - 1)) * tn_per + (in_xcd - tm_local * tn_per);
  if (tm_local >= tm_per || tile_m >= tiles_m || tile_n >= tiles_n) return;
  const int tile_id = tile_m * tiles_n + tile_n;
  const int m0 = tile_m * 32, n0 = tile_n * 32, z = PLAIN ? 0 : blockIdx.z;
  const __amdgpu_buffer_rsrc_t rsrc_a = small_rsrc(a.A + (int64_t)z * a.a_z_stride), rsrc_x = small_rsrc(a.X + (int64_t)z * a.x_z_stride);

  const int mrow = min(m0 + l32, a.M - 1);
  const int col = n0 + l32;
  const bool col_ok = col < a.Ncols;
  const int PQ = a.P * a.Q, HW = a.H * a.W, C = a.Kdim / 9;
  const float bias_c = 0.f;  // a per-column bias belongs to matrix products, which are never 3x3
  const int img = col_ok ? div_magic(col, PQ, a.magic_pq) : 0, pq = col_ok ? col - img * PQ : 0;
  const int p = div_magic(pq, a.Q, a.magic_q), q = pq - p * a.Q;
  const int ih0 = p * a.sh - a.ph, iw0 = q * a.sw - a.pw;
  // Half-wave h of iteration i takes channel cbeg + 2 i + h: the lane's offsets hold h, a tap's filter word or pixel and the mask
  // of what lies outside; the channel is in the scalar offset.
  unsigned x_off[9];
#pragma unroll
  for (int j = 0; j < 9; j++) {
    const int ih = ih0 + j / 3, iw = iw0 + j % 3;
    const bool ok = col_ok && (unsigned)ih < (unsigned)a.H && (unsigned)iw < (unsigned)a.W;
    x_off[j] = ok ? 4u * (unsigned)((int64_t)img * a.x_img_stride + half * HW + ih * a.W + iw) : SMALL_OUT_OF_RANGE;
  }
  const unsigned a_ch4 = 4u * 9u * (AMC ? (unsigned)a.a_ld : 1u), a_tap4 = 4u * (AMC ? (unsigned)a.a_ld : 1u);  // bytes between channels and taps
  const unsigned a_off = half * a_ch4 + 4u * (AMC ? (unsigned)mrow : (unsigned)mrow * (unsigned)a.Kdim);

  const int cbeg = ((int)blockIdx.y * KS + wave) * c_per_wave, cend = min(C, cbeg + c_per_wave);
  const int niter = max(0, (cend - cbeg + 1) >> 1);
  const bool odd = ((cend - cbeg) & 1) != 0;  // C is odd: the last iteration's second channel is none

  constexpr int DEPTH = 3;
  float ra[DEPTH][9], rb[DEPTH][9];
  auto load_iter = [&](int i, float (&av)[9], float (&bv)[9], auto last) {
    const unsigned c = (unsigned)(cbeg + 2 * i), as = c * a_ch4, xs = c * (unsigned)(4 * HW);
    // only the last iteration's lanes are masked, by an instruction a load
    const unsigned past = last && odd && i == niter - 1 ? (unsigned)half << 31 : 0u;
#pragma unroll
    for (int j = 0; j < 9; j++) {
      av[j] = small_load(rsrc_a, last ? a_off | past : a_off, as + j * a_tap4);
      bv[j] = small_load(rsrc_x, last ? x_off[j] | past : x_off[j], xs);
    }
  };

  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; r++) acc[r] = 0.f;
  Finish<KS> f;
  small_pipeline(niter, [&](int i, auto slot, auto last) { load_iter(i, ra[slot], rb[slot], last); },
                 [&](auto slot) {
#pragma unroll
                   for (int j = 0; j < 9; j++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[slot][j], rb[slot][j], acc, 0, 0, 0);
                 },
                 [&]() {
                   if constexpr (PLAIN) SMALL_LATE_ARGS();
                   prefetch_finish<KS>(a, z, m0, half, wave, img, pq, f);
                 });
  reduce_and_store<KS>(a, acc, f, bias_c, red, wave, lane, m0, img, pq, col_ok, z, (unsigned)(z * tiles + tile_id), splits, partials, counters);
#endif
}

// 1x1 geometry (convolution, possibly strided, or matrix product with A rows
// k-contiguous and B columns contiguous); Kdim % 4 == 0, A rows 16-byte aligned.
template <int KS, bool AMC, bool PLAIN>
__global__ __launch_bounds__(64 * KS) void conv1x1_f32_small_kernel(const float *A, const float *X, int M, int Ncols, int Kdim, int a_ld, int pixels,
                                                                    unsigned per_wave, unsigned magic_tn_per, unsigned magic_pq, const IgemmArgs args,
                                                                    int splits, float *partials, unsigned *counters) {
  #if __HIP_DEVICE_COMPILE__
  IgemmArgs a = small_args<PLAIN>(A, X, M, Ncols, Kdim, a_ld, 1, pixels, 1, per_wave, magic_tn_per, magic_pq, args);
  const int k_per_wave = (int)(per_wave >> 2);
  __shared__ float red[KS > 1 ? KS : 1][16][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, half = lane >> 5;
  // Workgroups go round-robin over the 8 XCDs (gridDim.x is a multiple of 8, so that holds for every y and
  // z as well), each with its own L2.  The XCDs are laid out as a grid of xcd_m x (8 / xcd_m) over the
  // (filter-row tile, column tile) plane and each owns one rectangle of tiles: it fetches 1 / xcd_m of the
  // filter and xcd_m / 8 of the activations, where a run of consecutive tiles per XCD fetches all of one operand
  // into all eight L2s.  The launcher picks xcd_m from the two operands' sizes.
  const int tiles_m = (a.M + 31) / 32, tiles_n = (a.Ncols + 31) / 32, tiles = tiles_n * tiles_m;
  const int tm_per = a.tm_per, tn_per = a.tn_per;
  const int xcd = (int)(blockIdx.x & 7), in_xcd = (int)(blockIdx.x >> 3);
  const int tm_local = div_magic(in_xcd, tn_per, a.magic_tn_per);
  const int tile_m = (xcd >> a.xcd_n_log2) * tm_per + tm_local;
  const int tile_n = (xcd & ((1 << a.xcd_n_log2) - 1)) * tn_per + (in_xcd - tm_local * tn_per);
  if (tm_local >= tm_per || tile_m >= tiles_m || tile_n >= tiles_n) return;
  const int tile_id = tile_m * tiles_n + tile_n;
  const int m0 = tile_m * 32, n0 = tile_n * 32, z = PLAIN ? 0 : blockIdx.z;
  // With a second convolution (a.A2) the reduction is the first's followed by the second's; a wavefront's slice
  // lies in one of them (the launcher makes k_per_wave divide Kdim), so it only picks its operands here.
  const int kbeg_all = ((int)blockIdx.y * KS + wave) * k_per_wave;
  const bool second = a.A2 != nullptr && kbeg_all >= a.Kdim;
  const __amdgpu_buffer_rsrc_t rsrc_a = small_rsrc(second ? a.A2 : a.A + (int64_t)z * a.a_z_stride),
                               rsrc_x = small_rsrc(second ? a.X2 : a.X + (int64_t)z * a.x_z_stride);
  const int Kd = second ? a.Kdim2 : a.Kdim;

  const int mrow = min(m0 + l32, a.M - 1);
  const int col = n0 + l32;
  const bool col_ok = col < a.Ncols;
  const int PQ = a.P * a.Q, HW = second ? a.H2 * a.W2 : a.H * a.W;
  const int img = col_ok ? div_magic(col, PQ, a.magic_pq) : 0, pq = col_ok ? col - img * PQ : 0;
  const int p = PLAIN ? 0 : div_magic(pq, a.Q, a.magic_q), q = pq - p * a.Q;
  const unsigned x_pix = second ? (unsigned)((int64_t)img * a.x2_img_stride + (int64_t)(p * a.sh2) * a.W2 + q * a.sw2)
                                : (unsigned)((int64_t)img * a.x_img_stride + (int64_t)(p * a.sh) * a.W + q * a.sw);
  // Half-wave h of iteration i takes k kbeg + 8 i + 4 h .. + 3 (Kd is a multiple of 4): h in the lane's offset, the rest in the scalar one.
  const unsigned x_k4 = 4u * (unsigned)HW, a_k4 = 4u * (AMC ? (unsigned)a.a_ld : 1u);
  const unsigned x_off = col_ok ? 4u * x_pix + 4u * half * x_k4 : SMALL_OUT_OF_RANGE;
  const unsigned a_off = 4u * half * a_k4 + 4u * (AMC ? (unsigned)mrow : (unsigned)mrow * (unsigned)Kd);

  const int kbeg = second ? kbeg_all - a.Kdim : kbeg_all, kend = min(Kd, kbeg + k_per_wave);
  const int niter = max(0, (kend - kbeg + 7) >> 3);
  const bool odd = ((kend - kbeg) & 7) != 0;  // the last iteration's second four k are none

  constexpr int DEPTH = 4;
  float4 ra[DEPTH];
  float rb[DEPTH][4];
  auto load_iter = [&](int i, float4 &av, float (&bv)[4]) {
    const unsigned k = (unsigned)(kbeg + 8 * i), as = k * a_k4, xs = k * x_k4;
    const unsigned past = odd && i == niter - 1 ? (unsigned)half << 31 : 0u;
    if (AMC) {
      av.x = small_load(rsrc_a, a_off | past, as); av.y = small_load(rsrc_a, a_off | past, as + a_k4);
      av.z = small_load(rsrc_a, a_off | past, as + 2u * a_k4); av.w = small_load(rsrc_a, a_off | past, as + 3u * a_k4);
    } else {
      av = small_load4(rsrc_a, a_off | past, as);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) bv[j] = small_load(rsrc_x, x_off | past, xs + j * x_k4);
  };

  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; r++) acc[r] = 0.f;
  auto mfma_iter = [&](int u) {
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[u].x, rb[u][0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[u].y, rb[u][1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[u].z, rb[u][2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[u].w, rb[u][3], acc, 0, 0, 0);
  };
  // Iteration i lives in slot i % DEPTH and is refilled with iteration i + DEPTH.  Whole groups that need every
  // refill run without a branch; the last DEPTH iterations refill nothing, and the group in between asks per
  // slot.  Most batch-1 layers have exactly DEPTH iterations per wavefront: everything is requested by the
  // prologue and nothing is loaded in vain.
  if (niter >= DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; d++) load_iter(d, ra[d], rb[d]);
  } else {
#pragma unroll
    for (int d = 0; d < DEPTH; d++)
      if (d < niter) load_iter(d, ra[d], rb[d]);
  }
  if constexpr (PLAIN) SMALL_LATE_ARGS();
  Finish<KS> f;
  prefetch_finish<KS>(a, z, m0, half, wave, img, pq, f);
  if (a.A2 != nullptr && a.bias2 != nullptr) {  // both biases ride in the one epilogue
#pragma unroll
    for (int i = 0; i < Finish<KS>::N; i++) f.bias[i] += a.bias2[min(acc_row(m0, half, wave * Finish<KS>::N + i), a.M - 1)];
  }
  const float bias_c = load_bias_col(a, col_ok ? col : 0);  // requested up front as well
  int i0 = 0;
  for (; i0 + 2 * DEPTH <= niter; i0 += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; u++) {
      mfma_iter(u);
      load_iter(i0 + u + DEPTH, ra[u], rb[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < DEPTH; u++) {
    if (i0 + u < niter) {
      mfma_iter(u);
      if (i0 + u + DEPTH < niter) load_iter(i0 + u + DEPTH, ra[u], rb[u]);
    }
  }
  i0 += DEPTH;
#pragma unroll
  for (int u = 0; u < DEPTH; u++)
    if (i0 + u < niter) mfma_iter(u);
  reduce_and_store<KS>(a, acc, f, bias_c, red, wave, lane, m0, img, pq, col_ok, z, (unsigned)(z * tiles + tile_id), splits, partials, counters);
#endif
}

// A fill kernel rather than hipMemsetAsync: a caller may be recording the stream into a graph.
__global__ void zero_counters_kernel(unsigned *counters, int n) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < n) counters[i] = 0u;
}

void clear_split_counters(const dnnrtContext *ctx, int n) {
  hipLaunchKernelGGL(zero_counters_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, ctx->stream, ctx->splitk_counters, n);
}

// Returns true if one of the specialised kernels took the problem.
bool launch_igemm_f32_small(const dnnrtContext *ctx, const IgemmArgs &a, int rsmode, int layout, bool &launched) {
  launched = false;
  if (layout != 0 && layout != 2) return true;
  const bool amc = layout == 2;
  // byte offsets below 2^31 inside the kernels
  const int64_t a_elems = amc ? (int64_t)a.Kdim * a.a_ld : (int64_t)a.M * a.Kdim;
  const int64_t x_elems = (int64_t)((a.Ncols + a.P * a.Q - 1) / (a.P * a.Q)) * a.x_img_stride + (int64_t)a.Kdim * a.H * a.W;
  if (a_elems >= (1ll << 29) || x_elems >= (1ll << 29)) return true;
  const bool is3x3 = rsmode == 3 && a.Kdim % 9 == 0 && !a.bias_col;
  const bool is1x1 = rsmode == 1 && (amc || a.a_vec4) && a.Kdim % 4 == 0 && a.Kdim >= 4;
  if (!is3x3 && !is1x1) return true;
  const bool dual = a.A2 != nullptr;
  if (dual) {
    const int64_t x2_elems = (int64_t)((a.Ncols + a.P * a.Q - 1) / (a.P * a.Q)) * a.x2_img_stride + (int64_t)a.Kdim2 * a.H2 * a.W2;
    if (!is1x1 || a.Z != 1 || a.Kdim2 % 8 != 0 || a.Kdim % 8 != 0 || x2_elems >= (1ll << 29) || (int64_t)a.Kdim2 * a.a_ld >= (1ll << 29) ||
        (int64_t)a.M * a.Kdim2 >= (1ll << 29))
      return true;
  }

  const int64_t tiles64 = ceil_div(a.M, 32) * ceil_div(a.Ncols, 32);
  if (tiles64 > INT32_MAX) return true;
  const int tiles = (int)tiles64;
  const int red_len = is3x3 ? a.Kdim / 9 : a.Kdim + (dual ? a.Kdim2 : 0);   // channels
  // reduction slice worth a wavefront; 1x1 problems of at most 32 tiles (the last stages of a MobileNetV2 at batch 1)
  // go down to 16 channels: 0.264 -> 0.260 ms per inference there, with more tiles it costs more than it gives
  const int min_slice = is3x3 ? SMALL_3X3_MIN_SLICE : (tiles <= 32 ? 16 : 32);
  int ks, splits;
  small_f32_cut(ctx->num_cu, (int64_t)tiles * a.Z, red_len, min_slice, ks, splits);
  if (splits > 1 && ((int64_t)tiles * a.Z * splits * 4096 > ctx->splitk_partial_bytes || (int64_t)tiles * a.Z > ctx->splitk_max_tiles)) {
    if (ctx->splitk_shared) {
      set_error("igemm_f32(small): the split reduction of this problem needs %lld bytes of scratch and %lld counters, "
                "the static scratch holds %lld and %d",
                (long long)tiles * a.Z * splits * 4096, (long long)tiles * a.Z, (long long)ctx->splitk_partial_bytes,
                ctx->splitk_max_tiles);
      return false;
    }
    // a handle's own scratch: a shallower split is as good
    while (splits > 1 && ((int64_t)tiles * a.Z * splits * 4096 > ctx->splitk_partial_bytes || (int64_t)tiles * a.Z > ctx->splitk_max_tiles)) splits /= 2;
  }
  int k_per_wave_1x1 = (int)(ceil_div(ceil_div(red_len, ks * splits), 8) * 8);
  if (dual) {
    // a slice must not straddle the two reductions: the next power of two, which has to divide the first one's
    // length (wavefronts whose slice starts past the end find every k masked)
    int p2 = 8;
    while (p2 < k_per_wave_1x1) p2 *= 2;
    if (a.Kdim % p2 != 0) return true;  // not launched: the caller runs the two convolutions one after the other
    k_per_wave_1x1 = p2;
  }
  // The XCD grid: xcd_m x (8 / xcd_m) rectangles of tiles.  Elements fetched over all eight L2s: the filter
  // 8 / xcd_m times, the activations xcd_m times; rectangles that do not divide the tile counts leave
  // workgroups without a tile and XCDs with less work, which the estimate charges for.
  IgemmArgs am = a;
  const int tiles_m = (int)ceil_div(a.M, 32), tiles_n = (int)ceil_div(a.Ncols, 32);
  int64_t slots = 0;
  {
    const double act = (double)(a.Kdim / (a.R * a.S)) * a.H * a.W * (double)ceil_div(a.Ncols, (int64_t)a.P * a.Q), filt = (double)a.M * a.Kdim;
    double best = 0;
    for (int xm = 1; xm <= 8; xm *= 2) {
      const int xn = 8 / xm;
      if ((xm > tiles_m && xm > 1) || (xn > tiles_n && xn > 1)) continue;
      const int64_t per = ceil_div(tiles_m, xm) * ceil_div(tiles_n, xn);
      const double cost = (act * xm + filt * xn) * ((double)(8 * per) / tiles);
      if (slots == 0 || cost < best) { best = cost; am.xcd_m = xm; slots = 8 * per; }
    }
    if (slots == 0) { am.xcd_m = 1; slots = 8 * ceil_div(tiles_m, 1) * ceil_div(tiles_n, 8); }  // a single tile either way
  }
  if (slots > INT32_MAX) return true;
  {
    const int xn = 8 / am.xcd_m;
    am.xcd_n_log2 = xn == 8 ? 3 : xn == 4 ? 2 : xn == 2 ? 1 : 0;
    am.tm_per = (int)ceil_div(tiles_m, am.xcd_m);
    am.tn_per = (int)ceil_div(tiles_n, xn);
    am.magic_tn_per = magic_of(am.tn_per);
    am.magic_pq = magic_of(a.P * a.Q);
    am.magic_q = magic_of(a.Q);
  }
  dim3 grid((unsigned)slots, splits, a.Z);
  if (ctx->splitk_shared && splits > 1) clear_split_counters(ctx, tiles * a.Z);
  const int per_wave = is3x3 ? (int)(ceil_div(ceil_div(red_len, ks * splits), 2) * 2) : k_per_wave_1x1;
  const unsigned per_wave_xn = 4u * (unsigned)per_wave + (unsigned)am.xcd_n_log2;
  const bool one_image = a.Ncols <= a.P * a.Q;  // of the images' distance nothing is read
  const bool plain = a.Z == 1 && !dual && a.sh == 1 && a.sw == 1 && a.P == a.H && a.Q == a.W && a.ph == (is3x3 ? 1 : 0) && a.pw == a.ph &&
                     (one_image || a.x_img_stride == (int64_t)(a.Kdim / (is3x3 ? 9 : 1)) * a.H * a.W);
#define LAUNCH_3X3(KS_, AMC_, PLAIN_)                                                                                                          \
  hipLaunchKernelGGL((conv3x3_f32_small_kernel<KS_, AMC_, PLAIN_>), grid, dim3(64 * KS_), 0, ctx->stream, a.A, a.X, a.M, a.Ncols, a.Kdim,       \
                     (int)a.a_ld, a.H, a.W, per_wave_xn, am.magic_tn_per, am.magic_pq, am.magic_q, am, splits, ctx->splitk_partials, ctx->splitk_counters)
#define LAUNCH_1X1(KS_, AMC_, PLAIN_)                                                                                                          \
  hipLaunchKernelGGL((conv1x1_f32_small_kernel<KS_, AMC_, PLAIN_>), grid, dim3(64 * KS_), 0, ctx->stream, a.A, a.X, a.M, a.Ncols, a.Kdim,       \
                     (int)a.a_ld, a.H * a.W, per_wave_xn, am.magic_tn_per, am.magic_pq, am, splits, ctx->splitk_partials, ctx->splitk_counters)
#define LAUNCH_KS(WHICH, AMC_, PLAIN_)          \
  switch (ks) {                                 \
    case 1: WHICH(1, AMC_, PLAIN_); break;      \
    case 2: WHICH(2, AMC_, PLAIN_); break;      \
    case 4: WHICH(4, AMC_, PLAIN_); break;      \
    default: WHICH(8, AMC_, PLAIN_); break;     \
  }
#define LAUNCH_AMC(WHICH, PLAIN_)                                                            \
  do {                                                                                       \
    if (amc) { LAUNCH_KS(WHICH, true, PLAIN_) } else { LAUNCH_KS(WHICH, false, PLAIN_) }     \
  } while (0)
  if (is3x3 && plain) LAUNCH_AMC(LAUNCH_3X3, true);
  else if (is3x3) LAUNCH_AMC(LAUNCH_3X3, false);
  else if (plain) LAUNCH_AMC(LAUNCH_1X1, true);
  else LAUNCH_AMC(LAUNCH_1X1, false);
#undef LAUNCH_AMC
#undef LAUNCH_KS
#undef LAUNCH_1X1
#undef LAUNCH_3X3
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("igemm_f32(small): launch failed: %s", hipGetErrorString(e)); return false; }
  launched = true;
  return true;
}

}  // namespace dnnrt
