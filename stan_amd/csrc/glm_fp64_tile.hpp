// Loads shared by the FP64 GLM passes.
#ifndef STANX_GLM_FP64_TILE_HPP
#define STANX_GLM_FP64_TILE_HPP

#include <hip/hip_runtime.h>

#include <cstdint>

#include "sx_internal.hpp"

namespace sx {
namespace {

// Buffer-resource loads: lanes whose offset is past `bytes` read zero and
// generate no memory request, so a tile's SMAX slot loads need no
// branches when the layout only holds S <= SMAX slots.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base,
                                                            uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0),
                                           static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ double buf_f64(__amdgpu_buffer_rsrc_t r, uint32_t voff,
                                          uint32_t soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 2));
}

// y of this lane's row (zero past N); issued before the tile's X loads so
// that waiting for it leaves the X loads in flight
template <int FAM>
__device__ __forceinline__ double load_y(const pass_args& a, int64_t t, int R, int r) {
  const int64_t row0 = t * R;
  const int64_t rows = a.N - row0 < R ? a.N - row0 : R;
  if (FAM == SX_LOGIT) {
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(static_cast<const int8_t*>(a.y) + row0, static_cast<uint32_t>(rows));
    return static_cast<double>(__builtin_amdgcn_raw_buffer_load_b8(rs, r, 0, 0));
  } else {
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(static_cast<const double*>(a.y) + row0, static_cast<uint32_t>(rows) * 8u);
    return buf_f64(rs, r * 8u, 0);
  }
}

}  // namespace
}  // namespace sx
#endif
