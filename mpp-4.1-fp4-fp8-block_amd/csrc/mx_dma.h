// mx_dma.h - global -> LDS loads through a buffer resource.
#pragma once

#include "mx_device.h"

namespace mx {

typedef __attribute__((address_space(3))) uint32_t* lds_u32;
extern "C" __device__ void llvm_amdgcn_raw_buffer_load_lds_u32(v4i rsrc, lds_u32 lds, int size, int voffset, int soffset,
                                                                int offset, int aux) __asm("llvm.amdgcn.raw.buffer.load.lds");

// `bytes` from base on (both uniform over the wave): loads past them read as
// zero.  FIRSTLANE: into scalar registers, where the compiler does not see that
// they are uniform.
template <bool FIRSTLANE>
__device__ __forceinline__ v4i rsrc_of(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  if constexpr (!FIRSTLANE) return v4i{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), (int)bytes, 0x00020000};
  v4i r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));
  r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
  r[3] = 0x00020000;
  return r;
}
__device__ __forceinline__ void buffer_dma16(v4i rsrc, void* lds, int offset) {
  llvm_amdgcn_raw_buffer_load_lds_u32(rsrc, (lds_u32)lds, 16, offset, 0, 0, 0);
}

}  // namespace mx
