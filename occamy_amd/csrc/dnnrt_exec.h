/* Entry points of the gfx950 runtime that the executor in this repository uses beside the C ABI of include/dnnrt.h.
 * They are looked up by name and may be missing (a host-only build has none): the executor then goes without. */
#pragma once
#include "../../include/dnnrt.h"

#ifdef __cplusplus
extern "C" {
#endif

/* An event that orders streams and keeps no time (dnnrtEventRecord, dnnrtEventDestroy). */
int32_t dnnrtExecFenceCreate(void **event);
/* What is issued on `stream` from now on starts after the work that `event` was last recorded behind. */
int32_t dnnrtExecStreamWait(dnnrtStream_t stream, void *event);

/* Copies pinned host memory to the device with a kernel: dst and src 16-byte aligned. */
int32_t dnnrtExecUpload(void *dst, const void *src, int64_t bytes, dnnrtStream_t stream);

/* An inverted residual block: y = act(conv1x1(actd(dwconv(act1(conv1x1(x, w1) + b1), wd) + bd), w3) + b3 [+ z]), square
 * stride, group of the middle convolution = its channels.  Rounded to fp16 where the separate calls round, behind each bias
 * and behind the sum with z; in front of that the fp32 sums start at the bias, which the separate calls add last, and run
 * in another order, so single results are another fp16 step than theirs.
 * fp16, N,H,W,C: w1 and w3 in blocks, dnnrtExecBlockFilter.  fp32, N,C,H,W, nothing rounded: wd C,R,S,K, w1 and w3 in
 * blocks, dnnrtExecBlockFilterF32. */
typedef struct dnnrtExecBlock {
  const void *x, *w1, *b1, *wd, *bd, *w3, *b3, *z; /* w1, b1: not read without expansion; z: residual laid out like y, or null */
  void *y;
  int64_t n, cin, h, w, ch, r, s, stride, pad_h, pad_w, p, q, cout;
  int64_t act1, actd, act; /* activation modes of the three convolutions and their coefficients */
  float coef1, coefd, coef;
  int32_t expand, dtype, format;
} dnnrtExecBlock;
/* 1 if dnnrtExecRunBlock takes the block (pointers aside) and is meant to be faster than the three calls. */
int32_t dnnrtExecBlockApplies(dnnrtHandle_t handle, const dnnrtExecBlock *block);
/* The layout of a 1x1 filter (rows x cols, fp16) for the block call, on the host: for every 32 rows, every 8 columns, the
 * rows' 8 values each. */
void dnnrtExecBlockFilter(void *dst, const void *src, int64_t rows, int64_t cols);
/* The same for fp32, from a filter C,R,S,K (cols x rows; cols is even): for every 16 rows, every two columns, the rows' two
 * values each. */
void dnnrtExecBlockFilterF32(void *dst, const void *src, int64_t rows, int64_t cols);
/* y must not overlap x or z. */
int32_t dnnrtExecRunBlock(dnnrtHandle_t handle, const dnnrtExecBlock *block);

#ifdef __cplusplus
}
#endif
