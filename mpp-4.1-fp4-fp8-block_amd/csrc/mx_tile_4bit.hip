// mx_tile_4bit.hip - prefill tile GEMM: f16 activations x MXFP4 or INT4 weights.
#include "mx_gemm_tile.h"

namespace mx {
namespace tile {

hipError_t launch_mxfp4(int side, int epi, const QGemmArgs& g, hipStream_t st) { return launch_f16a<BK_MXFP4>(side, epi, g, st); }
hipError_t launch_int4(int side, int epi, const QGemmArgs& g, hipStream_t st) { return launch_f16a<BK_INT4G32>(side, epi, g, st); }

}  // namespace tile
}  // namespace mx
