// mx_stream_8bit.hip - the weight-streaming GEMM's instances for 8-bit weights.
#include "mx_gemm_stream.h"

namespace mx {
namespace stream {

hipError_t launch_e4m3(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F16, BK_E4M3, false>(g, nullptr, 1, rows, ng, st);
}
hipError_t launch_e5m2(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F16, BK_E5M2, false>(g, nullptr, 1, rows, ng, st);
}
hipError_t launch_int8(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_F16, BK_INT8, false>(g, nullptr, 1, rows, ng, st);
}
hipError_t launch_i8(const Args& g, int rows, int ng, hipStream_t st) {
  return launch_bk<AK_I8, BK_I8, false>(g, nullptr, 1, rows, ng, st);
}

}  // namespace stream
}  // namespace mx
