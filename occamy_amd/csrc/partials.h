// Partial tiles of split reductions on their way between workgroups (igemm_f32_small.hip describes the hand-over): device-scope
// accesses, past the L2 of an XCD to the point where all of them agree, 16 bytes a lane (or eight, where a lane has no more).
// With four, and a part at a time, the last workgroup of a 64x64 tile in three parts issued 48 loads in three round trips: SRGAN
// at 90x117 (33 such layers) 675 -> 665 us, YOLO v1 794 -> 782, SSD300 1464 -> 1455, BERT fp16 568 -> 564.  Kernels on 32x32 tiles
// have two values a lane and did not move.
#pragma once
#include <hip/hip_runtime.h>

namespace dnnrt {

typedef float part_floatx4 __attribute__((ext_vector_type(4)));
typedef float part_floatx2 __attribute__((ext_vector_type(2)));

#if __HIP_DEVICE_COMPILE__
constexpr int PART_DEVICE_SCOPE = 16;           // cache policy sc1, as in a relaxed atomic access of agent scope
constexpr unsigned PART_NONE = 0x80000000u;     // offset of an access that is not made: a load of zeros
__device__ __forceinline__ __amdgpu_buffer_rsrc_t part_rsrc(float *partials) { return __builtin_amdgcn_make_buffer_rsrc(partials, 0, 0x7fffffff, 0x00020000); }
// voff: this lane's bytes, soff: uniform ones
__device__ __forceinline__ void part_store(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff, part_floatx4 v) {
  typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uintx4, v), r, (int)voff, (int)soff, PART_DEVICE_SCOPE);
}
__device__ __forceinline__ void part_store(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff, part_floatx2 v) {
  typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uintx2, v), r, (int)voff, (int)soff, PART_DEVICE_SCOPE);
}
template <class V>
__device__ __forceinline__ V part_load(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  if constexpr (sizeof(V) == 16) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, PART_DEVICE_SCOPE));
  else return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, PART_DEVICE_SCOPE));
}
#endif

}  // namespace dnnrt
