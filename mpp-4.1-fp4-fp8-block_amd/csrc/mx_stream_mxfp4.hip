// mx_stream_mxfp4.hip - the weight-streaming GEMM's instances for MXFP4 weights.
#include "mx_gemm_stream.h"

namespace mx {
namespace stream {

hipError_t launch_mxfp4(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F16, BK_MXFP4, false>(g, nullptr, 1, rows, ng, st);
}
hipError_t launch_f32_mxfp4(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F32, BK_MXFP4, false>(g, nullptr, 1, rows, ng, st);
}
hipError_t launch_mxfp4_grouped(const Args& g, const GroupTable& gt, int groups, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F16, BK_MXFP4, true>(g, &gt, groups, rows, ng, st);
}

}  // namespace stream
}  // namespace mx
