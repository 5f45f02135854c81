// fp16 matrix product (fp32 accumulate) on gfx950 MFMA.
#pragma once
#include "common.h"

namespace dnnrt {

struct GemmF16Args {
  const __half *A, *B, *C, *bias;
  __half *Out;
  int M, N, K;
  int64_t a_sm, a_sk, b_sk, b_sn;   // element strides of A along m and k, of B along k and n
  int64_t az, bz, yz;               // batch strides (0: shared)
  int64_t c_sm, cz;                 // C: row stride (0: one row for every m), batch stride
  float alpha, beta;
  int act;
  float act_coef;
  bool a_vec, b_vec;                // the contiguous direction of A / B may be read eight elements (16 bytes) at a time
  int steps_per_split;              // 64-k steps per workgroup along gridDim.y (the reduction split over workgroups)
  float *partials;                  // the handle's scratch: one 64 x 64 fp32 tile per (tile, split)
  unsigned *counters;               // ... and one arrival counter per tile, zero between kernels
};

// The product on tiles whose operands go straight into LDS (gemm_f16_dma.hip): row-major A, aligned rows; `launched` says
// whether it applied.  steps_per_split is set there.
bool launch_gemm_f16_dma(const dnnrtContext *ctx, const GemmF16Args &g, int Z, bool &launched);

// ... and on tiles whose four wavefronts share the reduction (gemm_f16_waves.hip); launch_gemm_f16_dma, its caller, has checked
// the forms.
bool launch_gemm_f16_waves(const dnnrtContext *ctx, const GemmF16Args &g, int Z, int rows, int splits);

// Out[z][M,N] = alpha * op(A[z]) op(B[z]) + beta * C[z]; strides in elements,
// 0 = operand shared by every z.
// bias: one value per column n, added to every row (may be null); act: an activation mode of apply_act applied last;
// C (scaled by beta) is a matrix like Out with the batch stride yz, or with c_is_row one row of N values.
bool gemm_f16(const dnnrtContext *ctx, const __half *A, const __half *B, const __half *C,
              __half *Out, int M, int N, int K, float alpha, float beta, bool transA, bool transB,
              int Z, int64_t az, int64_t bz, int64_t yz, bool c_is_row = false, const __half *bias = nullptr,
              int act = DNNRT_ACT_IDENTITY);

}  // namespace dnnrt
