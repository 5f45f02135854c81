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

#ifdef __cplusplus
}
#endif
