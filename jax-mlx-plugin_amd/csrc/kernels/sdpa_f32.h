// Loads shared by the fp32 matrix-core attention kernels (forward and
// backward): raw buffer resources that span exactly the valid rows of a tile,
// so rows past the end read as zeros and no load is predicated.
#pragma once

#include "sdpa_common.h"

namespace mfx {

// Bytes from the first to the last valid element of `rows` rows of D floats
// at `stride` floats apart (0 when no row is valid).
template <int D>
__device__ __forceinline__ int rows_extent(int rows, int64_t stride) {
  return rows > 0 ? (int)(((int64_t)(rows - 1) * stride + D) * 4) : 0;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t f32_rsrc(const float* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, bytes, 0x00020000);
}

__device__ __forceinline__ f32x4 ld4(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

}  // namespace mfx
