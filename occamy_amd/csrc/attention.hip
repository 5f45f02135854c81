// Multi-head attention core for transformer encoders:
//   Y[b, q, h*DH + d] = sum_k softmax_k(scale * <Q[b,q,h,:], K[b,k,h,:]>) * V[b,k,h,d]
// with Q, K, V, Y stored [batch, seq, heads * DH] (the layout the Linear layers
// write), fp32 or fp16 (a kernel each; everything between the fp16 tensors is
// in fp32, one rounding on the way out).  It stands for the chain the reference runs call by call --
// Reshape + Transpose of each operand (CUDAReshapeFunc, CUDATranspose4DFloatFunc),
// CUDAMatmulNdFunc, the scaling Mul, CUDASoftmaxFunc, CUDAMatmulNdFunc, Transpose
// + Reshape back -- twelve launches and eleven round trips through memory.
//
// fp32, many workgroups (attention_few_kernel takes the others): one workgroup = 32 queries of one head; its four wavefronts split every block
// of 128 keys (32 each).  Scores are computed transposed (keys x queries) so
// that a lane owns one query: the soft-max statistics are per lane, and the
// exponentiated scores already sit in the register layout the second product
// wants as its B operand (the 16 accumulator registers of a lane are 16 keys,
// which is just an ordering of the reduction index).  Keys are streamed in
// blocks with a running maximum and sum, so any sequence length works.
#include "common.h"

namespace dnnrt {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 att_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 att_half4 __attribute__((ext_vector_type(4)));
typedef short att_short4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float4 load4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ void store4(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }

// f of the two lanes that hold a query's keys, in both
template <typename F>
__device__ __forceinline__ float over_halves(float v, F f) {
#if __HIP_DEVICE_COMPILE__
  const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  v = f(__builtin_bit_cast(float, (unsigned)both[0]), __builtin_bit_cast(float, (unsigned)both[1]));
#endif
  return v;
}
__device__ __forceinline__ float max_over_halves(float v) {
  return over_halves(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float sum_over_halves(float v) {
  return over_halves(v, [](float a, float b) { return a + b; });
}

constexpr int ATT_QB = 32, ATT_KB = 128;

template <int DH>
__global__ __launch_bounds__(256) void attention_kernel(const float *__restrict__ Q, const float *__restrict__ K,
                                                        const float *__restrict__ V, float *__restrict__ Y, int Sq,
                                                        int Sk, int ld_in, int ld, float scale) {
  constexpr int ROW = DH + 4;       // LDS row stride in floats: 16-byte aligned rows, 16-byte reads spread over the banks
  constexpr int TD = DH / 32;       // 32-wide tiles of the head dimension
  extern __shared__ float smem[];
  float *Qs = smem;                 // [32][ROW]
  float *Ks = Qs + ATT_QB * ROW;    // [128][ROW]
  float *Vs = Ks + ATT_KB * ROW;    // [128][ROW]
  float *mx = Vs + ATT_KB * ROW;    // [4][32] block maxima per wavefront
  float *sm = mx + 4 * 32;          // [4][32] final sums per wavefront
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, half = lane >> 5;
  const int q0 = blockIdx.x * ATT_QB, head = blockIdx.y, b = blockIdx.z;
  const float *Qg = Q + (int64_t)b * Sq * ld_in + head * DH;
  const float *Kg = K + (int64_t)b * Sk * ld_in + head * DH;
  const float *Vg = V + (int64_t)b * Sk * ld_in + head * DH;

  // the query tile (rows past the end repeat the last query; they are not stored)
  // All of a tile's loads are requested before the first value goes to LDS (as a load-then-store loop the
  // compiler keeps one round trip to memory per turn: two for the queries, eight per block of keys and values,
  // most of the kernel's time at sequence length 128).
  constexpr int Q_TURNS = ATT_QB * (DH / 4) / 256, KV_TURNS = ATT_KB * (DH / 4) / 256, KV_CHUNK = KV_TURNS < 8 ? KV_TURNS : 8;
  static_assert(ATT_QB * (DH / 4) % 256 == 0 && ATT_KB * (DH / 4) % 256 == 0, "tile loads divide over the threads");
  {
    float4 qv[Q_TURNS];
#pragma unroll
    for (int u = 0; u < Q_TURNS; u++) {
      const int i = tid + 256 * u, r = i / (DH / 4), c4 = i - r * (DH / 4);
      qv[u] = load4(Qg + (int64_t)min(q0 + r, Sq - 1) * ld_in + c4 * 4);
    }
#pragma unroll
    for (int u = 0; u < Q_TURNS; u++) {
      const int i = tid + 256 * u, r = i / (DH / 4), c4 = i - r * (DH / 4);
      *reinterpret_cast<float4 *>(Qs + r * ROW + c4 * 4) = qv[u];
    }
  }

  floatx16 o[TD];
#pragma unroll
  for (int t = 0; t < TD; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[t][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  for (int kb = 0; kb < Sk; kb += ATT_KB) {
    __syncthreads();  // everyone is done with the previous block's K and V
#pragma unroll
    for (int u0 = 0; u0 < KV_TURNS; u0 += KV_CHUNK) {  // at most eight turns (64 registers) in flight
      float4 kv[KV_CHUNK], vv[KV_CHUNK];
#pragma unroll
      for (int u = 0; u < KV_CHUNK; u++) {
        const int i = tid + 256 * (u0 + u), r = i / (DH / 4), c4 = i - r * (DH / 4);
        const int64_t row = (int64_t)min(kb + r, Sk - 1) * ld_in + c4 * 4;
        kv[u] = load4(Kg + row);
        vv[u] = load4(Vg + row);
      }
#pragma unroll
      for (int u = 0; u < KV_CHUNK; u++) {
        const int i = tid + 256 * (u0 + u), r = i / (DH / 4), c4 = i - r * (DH / 4);
        *reinterpret_cast<float4 *>(Ks + r * ROW + c4 * 4) = kv[u];
        *reinterpret_cast<float4 *>(Vs + r * ROW + c4 * 4) = vv[u];
      }
      if (kb + ATT_KB > Sk)  // past the end the probability is zero, which times a repeated infinity would be NaN
#pragma unroll
        for (int u = 0; u < KV_CHUNK; u++) {
          const int i = tid + 256 * (u0 + u), r = i / (DH / 4), c4 = i - r * (DH / 4);
          if (kb + r >= Sk) *reinterpret_cast<float4 *>(Vs + r * ROW + c4 * 4) = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    __syncthreads();

    // scores, transposed: S[key][query] over this wavefront's 32 keys.  The
    // reduction index d is ordered so that lane half h walks d = h*DH/2 + i:
    // four consecutive MFMA operands are one 16-byte LDS read.
    floatx16 s;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.f;
    const float *krow = Ks + (wave * 32 + l32) * ROW + half * (DH / 2);
    const float *qrow = Qs + l32 * ROW + half * (DH / 2);
#pragma unroll
    for (int j = 0; j < DH / 8; j++) {
      const float4 ka = *reinterpret_cast<const float4 *>(krow + 4 * j);
      const float4 qa = *reinterpret_cast<const float4 *>(qrow + 4 * j);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(ka.x, qa.x, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(ka.y, qa.y, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(ka.z, qa.z, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(ka.w, qa.w, s, 0, 0, 0);
    }
    // register r of lane (l32, half) is key 8*(r/4) + 4*half + r%4 of the wavefront's 32, query l32
    float mloc = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int key = kb + wave * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
      s[r] = key < Sk ? s[r] * scale : -INFINITY;
      mloc = fmaxf(mloc, s[r]);
    }
    mloc = max_over_halves(mloc);
    if (half == 0) mx[wave * 32 + l32] = mloc;
    __syncthreads();
    const float mblk = fmaxf(fmaxf(mx[l32], mx[32 + l32]), fmaxf(mx[64 + l32], mx[96 + l32]));
    const float m_new = fmaxf(m_run, mblk);            // finite: every block holds at least one key
    const float alpha = expf(m_run - m_new);           // 0 on the first block
    float lsum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) { s[r] = expf(s[r] - m_new); lsum += s[r]; }
    l_run = l_run * alpha + lsum;                      // this lane's 16 keys; halves and wavefronts are added at the end
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < TD; t++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[t][r] *= alpha;
    // O^T[d][query] += V^T[d][key] * P^T[key][query]: step r takes, in lane
    // half h, key 8*(r/4) + 4*h + r%4 -- the key register r holds
    const float *vbase = Vs + (wave * 32 + 4 * half) * ROW + l32;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const float *vrow = vbase + (8 * (r >> 2) + (r & 3)) * ROW;
#pragma unroll
      for (int t = 0; t < TD; t++) o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * t], s[r], o[t], 0, 0, 0);
    }
  }

  // add the four wavefronts' partial outputs and sums, normalise, store
  __syncthreads();
  float *red = Ks;  // [4][32 queries][ROW], reusing the K and V tiles (4 * 32 rows <= 256 rows)
  l_run = sum_over_halves(l_run);
  if (half == 0) sm[wave * 32 + l32] = l_run;
#pragma unroll
  for (int t = 0; t < TD; t++)
#pragma unroll
    for (int g = 0; g < 4; g++)
      *reinterpret_cast<float4 *>(red + (wave * 32 + l32) * ROW + 32 * t + 8 * g + 4 * half) =
          make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
  __syncthreads();
  float *Yg = Y + (int64_t)b * Sq * ld + head * DH;
  for (int i = tid; i < ATT_QB * (DH / 4); i += 256) {
    const int q = i / (DH / 4), c4 = i - q * (DH / 4);
    if (q0 + q >= Sq) continue;
    const float inv = 1.0f / (sm[q] + sm[32 + q] + sm[64 + q] + sm[96 + q]);
    float4 acc = *reinterpret_cast<const float4 *>(red + q * ROW + c4 * 4);
#pragma unroll
    for (int w = 1; w < 4; w++) {
      const float4 p = *reinterpret_cast<const float4 *>(red + (w * 32 + q) * ROW + c4 * 4);
      acc.x += p.x; acc.y += p.y; acc.z += p.z; acc.w += p.w;
    }
    store4(Yg + (int64_t)(q0 + q) * ld + c4 * 4, make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv));
  }
}

// fp32, few workgroups: 16 queries of one head.  Its NW wavefronts take every NW-th block of 32 keys, each on its own, with its own
// running maximum and sum, and no barrier until the partial results meet.  All operands go straight from global memory into the shape of
// v_mfma_f32_16x16x4f32: a lane has the quarter (lane / 16) of the head dimension of its query and its keys, and of V the four
// keys of its quarter, whose probabilities are in its registers.  The next block's keys are requested behind the scores, its values
// behind the second product.
// Bound by the chain of one block: loads, half the 32-query kernel's MFMAs, exponentials, the meeting in LDS.  Back to back, against that
// kernel (us): 12 heads of 64, 128 tokens 7.0 -> 5.6, 32 tokens 7.1 -> 4.5, 256 tokens 11.0 -> 8.3, 16 queries over 512 keys 18.3 -> 11.2;
// 8 heads of 128, 128 tokens 10.5 -> 8.5.  Error against 64 bits 0.88 to 1.0 of that kernel's.  A BERT-base over 128 tokens 664 -> 641.
template <typename F>
__device__ __forceinline__ float over_quarters(float v, F f) {  // f of the four lanes that hold a query's keys, in all
#if __HIP_DEVICE_COMPILE__
  const auto rows = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  v = f(__builtin_bit_cast(float, (unsigned)rows[0]), __builtin_bit_cast(float, (unsigned)rows[1]));
#endif
  return over_halves(v, f);
}

template <int DH, int NW>
__global__ __launch_bounds__(64 * NW) void attention_few_kernel(const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V,
                                                                float *__restrict__ Y, int Sq, int Sk, int ld_in, int ld, float scale) {
#if __HIP_DEVICE_COMPILE__
  constexpr int T = DH / 16, ROW = DH + 4;
  __shared__ __attribute__((aligned(16))) float red[NW * 16 * ROW];
  __shared__ float mx[NW * 16], sm[NW * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, quarter = lane >> 4;
  const int q0 = blockIdx.x * 16, head = blockIdx.y, b = blockIdx.z;
  const float *Qg = Q + (int64_t)b * Sq * ld_in + head * DH + quarter * (DH / 4);
  const float *Kg = K + (int64_t)b * Sk * ld_in + head * DH + quarter * (DH / 4);
  const float *Vg = V + (int64_t)b * Sk * ld_in + head * DH + l16;
  float4 qf[T], kf[2][T];
  float vf[2][4][T];
  auto fetch_keys = [&](int k0) {  // rows past the end repeat the last key, masked below
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int j = 0; j < T; j++) kf[u][j] = load4(Kg + (int64_t)min(k0 + 16 * u + l16, Sk - 1) * ld_in + 4 * j);
  };
  auto fetch_values = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int t = 0; t < T; t++) vf[u][r][t] = Vg[(int64_t)min(k0 + 16 * u + 4 * quarter + r, Sk - 1) * ld_in + 16 * t];
  };
#pragma unroll
  for (int j = 0; j < T; j++) qf[j] = load4(Qg + (int64_t)min(q0 + l16, Sq - 1) * ld_in + 4 * j);
  floatx4 o[T];
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) o[t][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  int k0 = 32 * wave;
  if (k0 < Sk) { fetch_keys(k0); fetch_values(k0); }
  for (; k0 < Sk; k0 += 32 * NW) {
    floatx4 s[2];
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int r = 0; r < 4; r++) s[u][r] = 0.f;
#pragma unroll
    for (int j = 0; j < T; j++) {
#pragma unroll
      for (int u = 0; u < 2; u++) s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u][j].x, qf[j].x, s[u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < 2; u++) s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u][j].y, qf[j].y, s[u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < 2; u++) s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u][j].z, qf[j].z, s[u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < 2; u++) s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u][j].w, qf[j].w, s[u], 0, 0, 0);
    }
    const bool more = k0 + 32 * NW < Sk, last = k0 + 32 > Sk;
    if (more) fetch_keys(k0 + 32 * NW);
    // register r of s[u]: key k0 + 16 u + 4 quarter + r, query l16
    float m_new = m_run;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const bool in = !last || k0 + 16 * u + 4 * quarter + r < Sk;
        s[u][r] = in ? s[u][r] * scale : -INFINITY;
        m_new = fmaxf(m_new, s[u][r]);
      }
    m_new = over_quarters(m_new, [](float x, float y) { return fmaxf(x, y); });
    const float from = m_new == -INFINITY ? 0.f : m_new;  // this wavefront's keys alone may all have no weight
    const float alpha = expf(m_run - from);               // 0 on the first block
    float lsum = 0.f;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int r = 0; r < 4; r++) { s[u][r] = expf(s[u][r] - from); lsum += s[u][r]; }
    l_run = l_run * alpha + lsum;  // this lane's keys; the quarters and wavefronts are added at the end
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) o[t][r] *= alpha;
    if (last) {  // past the end the probability is zero, which times a repeated infinity would be NaN
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int t = 0; t < T; t++) vf[u][r][t] = k0 + 16 * u + 4 * quarter + r < Sk ? vf[u][r][t] : 0.f;
    }
    // O^T[d][query] += V^T[d][key] P^T[key][query]: step (u, r) takes, in lane quarter h, key 16 u + 4 h + r
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int t = 0; t < T; t++) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[u][r][t], s[u][r], o[t], 0, 0, 0);
    if (more) fetch_values(k0 + 32 * NW);
  }
  // the wavefronts' results: [NW][16 queries][ROW], their maxima and sums
  l_run = over_quarters(l_run, [](float x, float y) { return x + y; });
  if (quarter == 0) { mx[wave * 16 + l16] = m_run; sm[wave * 16 + l16] = l_run; }
#pragma unroll
  for (int t = 0; t < T; t++)
    store4(red + (wave * 16 + l16) * ROW + 16 * t + 4 * quarter, make_float4(o[t][0], o[t][1], o[t][2], o[t][3]));
  __syncthreads();
  float *Yg = Y + (int64_t)b * Sq * ld + head * DH;
  for (int i = tid; i < 16 * (DH / 4); i += 64 * NW) {
    const int q = i / (DH / 4), c = i - q * (DH / 4);
    if (q0 + q >= Sq) continue;
    float m = mx[q];
#pragma unroll
    for (int w = 1; w < NW; w++) m = fmaxf(m, mx[w * 16 + q]);
    float sum = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float f = expf(mx[w * 16 + q] - m);  // 0 for a wavefront that had no keys
      const float4 p = load4(red + (w * 16 + q) * ROW + 4 * c);
      sum += f * sm[w * 16 + q];
      acc.x += f * p.x; acc.y += f * p.y; acc.z += f * p.z; acc.w += f * p.w;
    }
    const float inv = 1.0f / sum;
    store4(Yg + (int64_t)(q0 + q) * ld + 4 * c, make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv));
  }
#endif
}

// exp(d) of a score below its maximum, d <= 0 or NaN, as 2^(d log2 e) with what the product rounds away put back to first order: half
// of expf's instructions, whose results below 2^-126 (here zero) the fp16 parts of a probability do not hold.
[[maybe_unused]] __device__ __forceinline__ float exp_of_score(float d) {
  constexpr float L_HI = 1.4426950216293335f, L_LO = 1.9259629911266175e-8f, LN2 = 0.69314718f;  // log2(e) in two parts
  d = __builtin_elementwise_maximum(d, -200.f);  // keeps NaN; -inf has no product to correct
  const float t = d * L_HI, rest = fmaf(d, L_LO, fmaf(d, L_HI, -t)), e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, rest * LN2, e);
}

// fp16.  A workgroup is 32 queries of one head; its NW wavefronts take every NW-th block of 32 keys, each on its own: its
// own running maximum and sum, no barrier until the partial results meet.  A block's scores are DH / 16 MFMAs of
// 32x32x16 (keys x queries, exact products, fp32 sums; K and Q straight from global memory in the operands' shape), and
// the register order of the scores is again the reduction order of the second product.  There the probabilities
// enter as two fp16 numbers each, p = hi + lo, scaled by 2^15: to within 2^-23 of themselves, or 2^-40 of the largest where
// that is more (with V at fp16's limits, a step of the smallest fp16 result); two MFMAs for what fp32 ones take eight times as
// long for.  Before its rounding the result is nearer to 64 bits than the fp32 kernel's on the same values: 384 keys, normal
// Q, K and V, relative error in the 2-norm at scales 0.001, 1/8, 1 and 4: 1.9e-7, 3.2e-7, 9.4e-7, 1.8e-6 -> 1.2e-7, 1.6e-7,
// 3.9e-7, 7.2e-7, and 0.25 to 1.0 of it over 16 to 2048 keys, head sizes 32 to 128, V positive or spread over 24 octaves (the
// scores' error decides, and their sums are shorter chains here).  A third part, all 24 bits, takes 1 % off that and adds 0.7
// us to 7.9.  V's operand, four consecutive keys of one d per read, comes out of the wavefront's LDS tile by transposing
// reads (ds_read_b64_tr_b16).
// Bound by latency (0.04 .. 0.8 GFLOP): 12 heads of 64, sequence 384: 19.3 us on fp32 MFMAs with fp16 storage -> 11.2 us
// (a pair of timestamps included in both); back to back 8.0 -> 7.2 us without a branch per load, with exp_of_score() and no masks
// but on the last block; 512 queries, 2048 keys, 4 heads: 22.8 -> 17.9.
// WIDE: rows are multiples of eight halfs apart, so sixteen bytes a load.  (Asked per load while running, the first loads alone were
// eleven branches, whose jumps cost more than the loads.)
template <int DH, int NW, bool WIDE>
__global__ __launch_bounds__(64 * NW) void attention_f16_kernel(const _Float16 *__restrict__ Q, const _Float16 *__restrict__ K,
                                                                const _Float16 *__restrict__ V, _Float16 *__restrict__ Y, int Sq,
                                                                int Sk, int ld_in, int ld, float scale) {
  constexpr int TD = DH / 32, SUB = DH / 16, VROW = DH + 8;  // V rows in LDS: 16-byte aligned, neighbouring rows in different banks
  constexpr int OROW = DH + 4;                               // rows of the partial results, floats
  constexpr int V_L = DH / 16;                               // 16-byte loads per lane for 32 rows of V
  extern __shared__ float smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, half = lane >> 5;
  const int q0 = blockIdx.x * 32, head = blockIdx.y, b = blockIdx.z;
  const _Float16 *Qg = Q + (int64_t)b * Sq * ld_in + head * DH;
  const _Float16 *Kg = K + (int64_t)b * Sk * ld_in + head * DH;
  const _Float16 *Vg = V + (int64_t)b * Sk * ld_in + head * DH;
  _Float16 *Vs = reinterpret_cast<_Float16 *>(smem) + wave * 32 * VROW;
  auto load8 = [&](const _Float16 *p) -> att_half8 {
    if constexpr (WIDE) return *reinterpret_cast<const att_half8 *>(p);
    const att_half4 lo = *reinterpret_cast<const att_half4 *>(p), hi = *reinterpret_cast<const att_half4 *>(p + 4);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  att_half8 qf[SUB], kf[SUB], vr[V_L];
#pragma unroll
  for (int s = 0; s < SUB; s++) qf[s] = load8(Qg + (int64_t)min(q0 + l32, Sq - 1) * ld_in + 16 * s + 8 * half);
  auto fetch = [&](int k0) {  // 32 keys from k0; rows past the end repeat the last key, masked below
    const _Float16 *krow = Kg + (int64_t)min(k0 + l32, Sk - 1) * ld_in + 8 * half;
#pragma unroll
    for (int s = 0; s < SUB; s++) kf[s] = load8(krow + 16 * s);
#pragma unroll
    for (int u = 0; u < V_L; u++) {
      const int i = lane + 64 * u, r = i / (DH / 8), c = i - r * (DH / 8);
      vr[u] = load8(Vg + (int64_t)min(k0 + r, Sk - 1) * ld_in + 8 * c);
    }
  };
  floatx16 o[TD];
#pragma unroll
  for (int t = 0; t < TD; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[t][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  int k0 = 32 * wave;
  if (k0 < Sk) fetch(k0);
  for (; k0 < Sk; k0 += 32 * NW) {
    floatx16 s;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.f;
#pragma unroll
    for (int u = 0; u < SUB; u++) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[u], qf[u], s, 0, 0, 0);
    asm volatile("" ::: "memory");  // the transposing reads of the block before are behind us
#pragma unroll
    for (int u = 0; u < V_L; u++) {
      const int i = lane + 64 * u, r = i / (DH / 8), c = i - r * (DH / 8);
      *reinterpret_cast<att_half8 *>(Vs + r * VROW + 8 * c) = vr[u];
    }
    asm volatile("" ::: "memory");  // a wavefront's LDS accesses are carried out in order
    if (k0 + 32 * NW < Sk) fetch(k0 + 32 * NW);
    // register r of lane (l32, half): key k0 + 8 * (r / 4) + 4 * half + r % 4, query l32
    float m_new = m_run;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] *= scale;
    if (k0 + 32 > Sk) {
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] = k0 + 8 * (r >> 2) + 4 * half + (r & 3) < Sk ? s[r] : -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; r++) m_new = fmaxf(m_new, s[r]);
    m_new = max_over_halves(m_new);  // finite: every block that is entered holds a key
    const float alpha = expf(m_run - m_new);          // 0 on the first block
    float lsum = 0.f;
    att_half8 hi[2], lo[2];
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const float p = exp_of_score(s[r] - m_new) * 32768.f;
      lsum += p;
      const _Float16 h = (_Float16)p;
      hi[r >> 3][r & 7] = h;
      lo[r >> 3][r & 7] = (_Float16)(p - (float)h);
    }
    l_run = l_run * alpha + lsum;  // this lane's keys; the halves are added at the end
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < TD; t++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[t][r] *= alpha;
    // O^T[d][query] += V^T[d][key] P^T[key][query]: element e of lane half h is key 16 u + 8 (e / 4) + 4 h + e % 4
#if __HIP_DEVICE_COMPILE__
    typedef __attribute__((address_space(3))) att_short4 *tr_ptr;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int t = 0; t < TD; t++) {
        const _Float16 *at = Vs + (16 * u + 4 * half + ((lane & 15) >> 2)) * VROW + 32 * t + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        const att_short4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)at), v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + 8 * VROW));
        const att_half8 vf = __builtin_bit_cast(att_half8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, hi[u], o[t], 0, 0, 0);
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, lo[u], o[t], 0, 0, 0);
      }
#endif
  }
  // the wavefronts' results: [NW][32 queries][OROW], then maxima and sums [NW][32] each
  __syncthreads();
  float *red = smem, *mx = red + NW * 32 * OROW, *sm = mx + NW * 32;
  l_run = sum_over_halves(l_run);
  if (half == 0) { mx[wave * 32 + l32] = m_run; sm[wave * 32 + l32] = l_run; }
#pragma unroll
  for (int t = 0; t < TD; t++)
#pragma unroll
    for (int g = 0; g < 4; g++)
      store4(red + (wave * 32 + l32) * OROW + 32 * t + 8 * g + 4 * half, make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]));
  __syncthreads();
  _Float16 *Yg = Y + (int64_t)b * Sq * ld + head * DH;
  for (int i = tid; i < 32 * (DH / 8); i += 64 * NW) {
    const int q = i / (DH / 8), c = i - q * (DH / 8);
    if (q0 + q >= Sq) continue;
    float m = mx[q];
#pragma unroll
    for (int w = 1; w < NW; w++) m = fmaxf(m, mx[w * 32 + q]);
    float sum = 0.f, v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float f = expf(mx[w * 32 + q] - m);  // 0 for a wavefront that had no keys
      sum += f * sm[w * 32 + q];
      const float4 a = load4(red + (w * 32 + q) * OROW + 8 * c), d = load4(red + (w * 32 + q) * OROW + 8 * c + 4);
      v[0] += f * a.x; v[1] += f * a.y; v[2] += f * a.z; v[3] += f * a.w;
      v[4] += f * d.x; v[5] += f * d.y; v[6] += f * d.z; v[7] += f * d.w;
    }
    // An infinity in V may have met a part of a probability that is zero or negative and left NaN.  Probabilities are positive
    // and finite where their sum is, so the column's infinities alone are the result (and a NaN in V stays one).
    bool finite = true;
#pragma unroll
    for (int e = 0; e < 8; e++) finite = finite && fabsf(v[e]) < INFINITY;
    if (!finite && sum < INFINITY) {
      float t[8] = {};
      for (int key = 0; key < Sk; key++) {
        const att_half8 x = load8(Vg + (int64_t)key * ld_in + 8 * c);
#pragma unroll
        for (int e = 0; e < 8; e++) t[e] += (float)x[e];  // the finite ones' sum is finite
      }
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] = fabsf(t[e]) < INFINITY ? v[e] : t[e];
    }
    const float inv = 1.0f / sum;
    att_half8 out;
#pragma unroll
    for (int e = 0; e < 8; e++) out[e] = (_Float16)(v[e] * inv);
    *reinterpret_cast<att_half8 *>(Yg + (int64_t)(q0 + q) * ld + 8 * c) = out;
  }
}

template <int DH>
static void launch_attention(const dnnrtContext *ctx, const float *Q, const float *K, const float *V, float *Y, int B,
                             int Sq, int Sk, int H, int ld_in, float scale) {
  // While 16 queries a workgroup are no more than one per compute unit; beyond, the 32-query kernel reads K and V half as often: 384
  // tokens, 12 heads 16.0 here, 15.2 there; 4 x 128 tokens 8.8, 7.3 (one long sequence, 1024 tokens, 48.5 and 54.9, is the exception).
  if (ceil_div(Sq, 16) * H * B <= (int64_t)ctx->num_cu) {
    constexpr int MORE = DH <= 64 ? 8 : 4;
    const dim3 grid((unsigned)ceil_div(Sq, 16), (unsigned)H, (unsigned)B);
    if (Sk > 128) hipLaunchKernelGGL((attention_few_kernel<DH, MORE>), grid, dim3(64 * MORE), 0, ctx->stream, Q, K, V, Y, Sq, Sk, ld_in, H * DH, scale);
    else hipLaunchKernelGGL((attention_few_kernel<DH, 4>), grid, dim3(256), 0, ctx->stream, Q, K, V, Y, Sq, Sk, ld_in, H * DH, scale);
    return;
  }
  constexpr int ROW = DH + 4;
  const size_t lds = (size_t)((ATT_QB + 2 * ATT_KB) * ROW + 8 * 32) * sizeof(float);
  static LdsRaised raised;
  (void)raise_lds(raised, ctx->device, reinterpret_cast<const void *>(&attention_kernel<DH>), (int)lds);  // refused: the launch says so
  hipLaunchKernelGGL((attention_kernel<DH>), dim3((unsigned)ceil_div(Sq, ATT_QB), (unsigned)H, (unsigned)B), dim3(256),
                     lds, ctx->stream, Q, K, V, Y, Sq, Sk, ld_in, H * DH, scale);
}

template <int DH, int NW, bool WIDE>
static void launch_attention_f16(const dnnrtContext *ctx, const __half *Q, const __half *K, const __half *V, __half *Y, int B,
                                 int Sq, int Sk, int H, int ld_in, float scale) {
  const size_t lds = (size_t)NW * 32 * (DH + 4 + 2) * sizeof(float);  // the partial results; the V tiles lie under them
  static_assert((DH + 8) * 2 <= (DH + 4) * 4, "V tiles fit");
  static LdsRaised raised;
  (void)raise_lds(raised, ctx->device, reinterpret_cast<const void *>(&attention_f16_kernel<DH, NW, WIDE>), (int)lds);
  hipLaunchKernelGGL((attention_f16_kernel<DH, NW, WIDE>), dim3((unsigned)ceil_div(Sq, 32), (unsigned)H, (unsigned)B), dim3(64 * NW), lds, ctx->stream,
                     (const _Float16 *)Q, (const _Float16 *)K, (const _Float16 *)V, (_Float16 *)Y, Sq, Sk, ld_in, H * DH, scale);
}

template <int DH>
static void launch_attention(const dnnrtContext *ctx, const __half *Q, const __half *K, const __half *V, __half *Y, int B,
                             int Sq, int Sk, int H, int ld_in, float scale) {
  // eight wavefronts where four would leave SIMDs idle and there are keys for more
  const bool more = DH <= 64 && Sk > 128 && ceil_div(Sq, 32) * H * B < 2 * (int64_t)ctx->num_cu;
  constexpr int MORE = DH <= 64 ? 8 : 4;
  if (ld_in % 8 == 0) {
    if (more) launch_attention_f16<DH, MORE, true>(ctx, Q, K, V, Y, B, Sq, Sk, H, ld_in, scale);
    else launch_attention_f16<DH, 4, true>(ctx, Q, K, V, Y, B, Sq, Sk, H, ld_in, scale);
  } else {
    if (more) launch_attention_f16<DH, MORE, false>(ctx, Q, K, V, Y, B, Sq, Sk, H, ld_in, scale);
    else launch_attention_f16<DH, 4, false>(ctx, Q, K, V, Y, B, Sq, Sk, H, ld_in, scale);
  }
}

}  // namespace dnnrt

using namespace dnnrt;

extern "C" void *dnnrtAttention(dnnrtHandle_t handle, const void *Q, const void *K, const void *V, void *Y,
                                int64_t batch, int64_t seqQ, int64_t seqK, int64_t heads, int64_t headDim,
                                int64_t ldIn, float scale, int32_t dtype) {
  if (!handle) DNNRT_FAIL("dnnrtAttention: null handle");
  if (!Q || !K || !V || !Y) DNNRT_FAIL("dnnrtAttention: null argument");
  if (dtype != DNNRT_F32 && dtype != DNNRT_F16) DNNRT_FAIL("dnnrtAttention: dtype %d (fp32 and fp16)", dtype);
  if (batch < 0 || seqQ < 0) DNNRT_FAIL("dnnrtAttention: bad dims");
  if (batch == 0 || seqQ == 0) return Y;  // no queries: no work
  if (seqK <= 0 || heads <= 0) DNNRT_FAIL("dnnrtAttention: bad dims");
  if (batch > 65535 || heads > 65535 || seqQ > (1 << 24) || seqK > (1 << 24)) DNNRT_FAIL("dnnrtAttention: dims too large");
  if (headDim != 32 && headDim != 64 && headDim != 128) DNNRT_FAIL("dnnrtAttention: head dim %ld (32, 64, 128)", (long)headDim);
  if (!aligned16(Q) || !aligned16(K) || !aligned16(V) || !aligned16(Y)) DNNRT_FAIL("dnnrtAttention: operands must be 16-byte aligned");
  if (Y == Q || Y == K || Y == V) DNNRT_FAIL("dnnrtAttention: Y must not alias an input");
  if (ldIn == 0) ldIn = heads * headDim;
  if (ldIn < heads * headDim || ldIn % 4 || ldIn > INT32_MAX) DNNRT_FAIL("dnnrtAttention: ldIn %ld (>= heads * headDim, multiple of 4)", (long)ldIn);
  auto run = [&](auto *q, auto *k, auto *v, auto *y) {
    if (headDim == 32) launch_attention<32>(handle, q, k, v, y, (int)batch, (int)seqQ, (int)seqK, (int)heads, (int)ldIn, scale);
    else if (headDim == 64) launch_attention<64>(handle, q, k, v, y, (int)batch, (int)seqQ, (int)seqK, (int)heads, (int)ldIn, scale);
    else launch_attention<128>(handle, q, k, v, y, (int)batch, (int)seqQ, (int)seqK, (int)heads, (int)ldIn, scale);
  };
  if (dtype == DNNRT_F32) run((const float *)Q, (const float *)K, (const float *)V, (float *)Y);
  else run((const __half *)Q, (const __half *)K, (const __half *)V, (__half *)Y);
  DNNRT_CHECK_LAUNCH("dnnrtAttention");
  return Y;
}
