// mx_tile_16.hip - prefill tile GEMM: f16 x f16 and int8 x int8 (W8A8).
#include "mx_gemm_tile.h"

namespace mx {
namespace tile {

hipError_t launch_f16(int side, int epi, const QGemmArgs& g, hipStream_t st) { return launch_f16a<BK_F16>(side, epi, g, st); }

hipError_t launch_i8(int epi, const QGemmArgs& g, hipStream_t st) {
  switch (epi) {
    case EPI_SWIGLU_F32: return launch_one<AK_I8, BK_I8, EPI_SWIGLU_F32, 256>(g, st);
    case EPI_STORE_F16: return launch_one<AK_I8, BK_I8, EPI_STORE_F16, 256>(g, st);
    case EPI_STORE_F32: return launch_one<AK_I8, BK_I8, EPI_STORE_F32, 256>(g, st);
    case EPI_STORE_I32: return launch_one<AK_I8, BK_I8, EPI_STORE_I32, 256>(g, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tile
}  // namespace mx
