// mx_tile_8bit.hip - prefill tile GEMM: f16 activations x FP8 or INT8 weights.
#include "mx_gemm_tile.h"

namespace mx {
namespace tile {

hipError_t launch_e4m3(int side, int epi, const QGemmArgs& g, hipStream_t st) { return launch_f16a<BK_E4M3>(side, epi, g, st); }
hipError_t launch_e5m2(int side, int epi, const QGemmArgs& g, hipStream_t st) { return launch_f16a<BK_E5M2>(side, epi, g, st); }
hipError_t launch_int8(int side, int epi, const QGemmArgs& g, hipStream_t st) { return launch_f16a<BK_INT8>(side, epi, g, st); }

}  // namespace tile
}  // namespace mx
