// Helpers shared by the kernels that stage K and V tiles of 16-bit elements in
// LDS (rbf_tile_impl.h, rbf_block_impl.h).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vectra {

// Whether a 16-byte chunk of T holds only finite values.
template <typename T>
__device__ __forceinline__ bool finite_chunk(const uint4& r) {
  constexpr uint32_t kExp = __is_same(T, __bf16) ? 0x7f80u : 0x7c00u;
  const uint32_t w[4] = {r.x, r.y, r.z, r.w};
  bool finite = true;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    finite = finite && (w[e] & kExp) != kExp && (w[e] & (kExp << 16)) != (kExp << 16);
  return finite;
}

}  // namespace vectra
