// mx_stream_f16.hip - the weight-streaming GEMM's instances for f16 and INT4 weights.
#include "mx_gemm_stream.h"

namespace mx {
namespace stream {

hipError_t launch_f16(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F16, BK_F16, false>(g, nullptr, 1, rows, ng, st);
}
hipError_t launch_f32_f16(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F32, BK_F16, false>(g, nullptr, 1, rows, ng, st);
}
hipError_t launch_int4(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F16, BK_INT4G32, false>(g, nullptr, 1, rows, ng, st);
}

}  // namespace stream
}  // namespace mx
